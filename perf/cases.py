"""The work that programs using this library have it do, as timed cases.

Every case goes through a public entry point of the Python package and stands
for a kind of call over a range of sizes:

  convolve   one device-resident circular convolution (``convolve3d``)
  correlate  its adjoint with respect to the image (``op=CORRELATE``)
  boundary   linear convolution of an extended image (``convolve3d_boundary``)
  plan       one PSF applied to image after image (``ConvolutionPlan.run``)
  train      forward and both gradients through torch autograd
  batch      many uneven blocks through one ``BatchedConvolution``
  rl         multiview Richardson-Lucy deconvolution
  host       the drop-in call on host buffers, in place

``listed()`` gives the named cases, ``draw(rng)`` one more of the same ranges:
image extents from 48 to 640 in x and y and from 24 to 320 in z, half of them
the extents volumes are commonly cut to and half any integer (stacks are
cropped and padded to whatever a specimen needs), PSF extents from 5 to 41
(91 along z).  Sizes are given as {x, y, z} like the library's C interface.
"""
import math

import numpy as np
import torch

import fourierconvolutioncudalib_amd as fc
from fourierconvolutioncudalib_amd import synth
from fourierconvolutioncudalib_amd.autograd import fft_conv3d
from fourierconvolutioncudalib_amd.batched import BatchedConvolution
from fourierconvolutioncudalib_amd.rl import richardson_lucy


def _case(kind, n, k, **more):
    return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], kx=k[0], ky=k[1], kz=k[2], **more)


def listed():
    return [
        # a small block with a compact PSF: launches and host time count
        _case("convolve", (64, 64, 64), (7, 7, 7), name="convolve_64x64x64"),
        # a region of interest
        _case("convolve", (128, 128, 64), (15, 15, 15), name="convolve_128x128x64"),
        # one camera stack, the benchmark's volume
        _case("convolve", (512, 512, 256), (15, 15, 15), name="convolve_512x512x256"),
        # a light-sheet stack with a long axial PSF, the largest volume
        _case("convolve", (600, 500, 240), (31, 31, 61), name="convolve_600x500x240"),
        # stacks padded by their PSF's extents, so extents with large prime factors
        _case("convolve", (158, 158, 218), (31, 31, 91), name="convolve_158x158x218"),
        _case("correlate", (286, 286, 346), (31, 31, 91), name="correlate_286x286x346"),
        # one PSF, image after image
        _case("plan", (384, 384, 192), (25, 25, 51), name="plan_384x384x192"),
        # a stack whose edges must not wrap around
        _case("boundary", (512, 512, 256), (15, 15, 15), mode="reflect",
              name="boundary_reflect_512x512x256"),
        # fitting an image and a PSF by gradient descent
        _case("train", (256, 256, 128), (21, 21, 21), name="train_256x256x128"),
        # uneven blocks, each with its own PSF
        dict(kind="batch", count=24, shapes=3003, ragged=False, name="batch_24_blocks"),
        # four views fused into one estimate
        _case("rl", (384, 384, 192), (25, 25, 51), views=4, iterations=10, name="rl_4x384x384x192"),
        # the drop-in call of an existing host program
        _case("host", (256, 256, 128), (15, 15, 15), name="host_256x256x128"),
    ]


# extents that volumes are commonly cut to
_COMMON = (48, 64, 80, 96, 100, 112, 120, 128, 144, 160, 192, 200, 224, 240, 256, 288, 300, 320,
           384, 400, 448, 480, 512, 576, 600, 640)


def _extent(rng, lo, hi):
    n = round(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    if rng.random() < 0.5:
        n = min((c for c in _COMMON if lo <= c <= hi), key=lambda c: abs(math.log(c / n)))
    return n


def _taps(rng, hi, n):
    k = rng.randint(5, hi)
    if k % 2 == 0 and rng.random() < 0.8:  # most PSFs have a centre voxel
        k += 1
    return min(k, n)


def draw(rng):
    kind = rng.choice(("convolve",) * 4 + ("correlate", "boundary", "boundary", "plan", "plan",
                                           "train", "train", "batch", "rl", "host"))
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(6, 24), shapes=rng.randint(1, 9999),
                    ragged=rng.random() < 0.5)
    most = {"rl": 16e6, "host": 32e6, "train": 32e6, "boundary": 48e6}.get(kind, 72e6)
    while True:
        n = (_extent(rng, 48, 640), _extent(rng, 48, 640), _extent(rng, 24, 320))
        if n[0] * n[1] * n[2] <= most:
            break
    k = (_taps(rng, 41, n[0]), _taps(rng, 41, n[1]), _taps(rng, 91, n[2]))
    if kind == "boundary":
        return _case(kind, n, k, mode=rng.choice(("zero", "nearest", "reflect", "mirror")))
    if kind == "rl":
        return _case(kind, n, k, views=rng.randint(1, 4), iterations=rng.randint(2, 10))
    return _case(kind, n, k)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _block_shapes(case):
    """[(image shape, PSF shape, PSF seed)], C order."""
    if not case["ragged"]:
        return synth.uneven_block_shapes(case["shapes"], case["count"])
    return synth.uneven_block_shapes(case["shapes"], case["count"], menu=tuple(range(64, 257)))


def _stack(shape, gen, noise=True):
    """A light-sheet-like stack: bright structures a few voxels wide on a
    dark background, with photon noise."""
    coarse = torch.rand([1, 1] + [max(2, n // 6) for n in shape], device="cuda", generator=gen)
    v = torch.nn.functional.interpolate(coarse, size=shape, mode="trilinear")[0, 0]
    v = 20.0 + 900.0 * v.pow(6)
    return (torch.poisson(v, generator=gen) if noise else v).contiguous()


def _psf(case, seed, view=0):
    k = (case["kz"], case["ky"], case["kx"])
    r = np.random.default_rng([seed, view])
    sigma = [max(0.6, n / 8.0) * r.uniform(0.9, 1.1) for n in k[::-1]]
    turn = synth.rotation_y(180.0 * view / case.get("views", 1)) if view else None
    return torch.from_numpy(synth.gaussian_psf(k, sigma, turn)).cuda()


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "batch":
        spec = _block_shapes(case)
        images = [_stack(s, gen) for s, _, _ in spec]
        psfs = [torch.from_numpy(synth.random_psf(k, p + seed)).cuda() for _, k, p in spec]
        return dict(kind=kind, images=images, psfs=psfs, plan=BatchedConvolution(images, psfs))
    shape = (case["nz"], case["ny"], case["nx"])
    if kind == "rl":
        views = [_stack(shape, gen) for _ in range(case["views"])]
        psfs = [_psf(case, seed, v) for v in range(case["views"])]
        return dict(kind=kind, views=views, psfs=psfs, iterations=case["iterations"])
    image, psf = _stack(shape, gen), _psf(case, seed)
    state = dict(kind=kind, image=image, psf=psf)
    if kind == "host":
        return dict(kind=kind, image=image.cpu().numpy().reshape(-1), n=list(shape[::-1]),
                    psf=psf.cpu().numpy().reshape(-1), k=[case["kx"], case["ky"], case["kz"]])
    if kind == "boundary":
        state["mode"] = case["mode"]
    if kind == "plan":
        state["plan"] = fc.ConvolutionPlan(shape, psf)
        state["out"] = torch.empty_like(image)
    if kind == "train":
        state["grad"] = torch.randn(shape, device="cuda", generator=gen)
        image.requires_grad_(True)
        psf.requires_grad_(True)
    return state


def run(state):
    kind = state["kind"]
    if kind == "convolve":
        return fc.convolve3d(state["image"], state["psf"])
    if kind == "correlate":
        return fc.convolve3d(state["image"], state["psf"], op=fc.CORRELATE)
    if kind == "boundary":
        return fc.convolve3d_boundary(state["image"], state["psf"], state["mode"])
    if kind == "plan":
        return state["plan"].run(state["image"], out=state["out"])
    if kind == "train":
        out = fft_conv3d(state["image"], state["psf"])
        gi, gk = torch.autograd.grad(out, (state["image"], state["psf"]), state["grad"])
        return {"out": out.detach(), "grad_image": gi, "grad_psf": gk}
    if kind == "batch":
        return state["plan"].run()
    if kind == "rl":
        return richardson_lucy(state["views"], state["psfs"], state["iterations"])
    fc.convolution3DfftCUDAInPlace(state["image"], state["n"], state["psf"], state["k"], 0)
    return state["image"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _conv_work(n, k):
    """Bytes: image and PSF read once, result written once.  Operations: a
    real transform forth and back and the product."""
    v = n[0] * n[1] * n[2]
    return 8 * v + 4 * k[0] * k[1] * k[2], 5 * v * math.log2(v) + 3 * v


def work(case):
    if case["kind"] == "batch":
        each = [_conv_work(s, k) for s, k, _ in _block_shapes(case)]
        return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}
    n, k = (case["nx"], case["ny"], case["nz"]), (case["kx"], case["ky"], case["kz"])
    v, taps = n[0] * n[1] * n[2], k[0] * k[1] * k[2]
    b, f = _conv_work(n, k)
    if case["kind"] == "train":  # image, PSF and gradient in; result and two gradients out
        return {"bytes": 16 * v + 8 * taps, "flops": 2.5 * f}
    if case["kind"] == "rl":  # the views and PSFs in, the estimate out
        return {"bytes": 4 * (v + taps) * case["views"] + 4 * v,
                "flops": 2 * f * case["views"] * case["iterations"]}
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _spectrum(psf, shape):
    """Half spectrum of the PSF placed circularly, its centre k // 2 at 0."""
    grid = torch.zeros(shape, dtype=torch.float64, device=psf.device)
    z, y, x = ((torch.arange(k, device=psf.device) - k // 2) % n for k, n in zip(psf.shape, shape))
    grid[z[:, None, None], y[None, :, None], x[None, None, :]] = psf.double()
    return torch.fft.rfftn(grid)


def _filter(image, spectrum, adjoint=False):
    s = torch.fft.rfftn(image.double())
    s *= spectrum.conj() if adjoint else spectrum
    return torch.fft.irfftn(s, s=image.shape)


def _source(p, n, mode):
    """Index of element p (an int64 tensor) of the extended axis, and where it is not zero."""
    inside = (p >= 0) & (p < n)
    if mode == "zero":
        return p.clamp(0, n - 1), inside
    if mode == "nearest":
        return p.clamp(0, n - 1), torch.ones_like(inside)
    period = 2 * n if mode == "reflect" else max(1, 2 * n - 2)
    r = p % period
    return torch.where(r < n, r, period - (1 if mode == "reflect" else 0) - r), torch.ones_like(inside)


def _extended(image, kshape, mode):
    v = image.double()
    for axis, (n, k) in enumerate(zip(image.shape, kshape)):
        p = torch.arange(n + k - 1, device=image.device) - (k - 1 - k // 2)
        index, ok = _source(p, n, mode)
        v = v.index_select(axis, index)
        v *= ok.double().reshape([-1 if a == axis else 1 for a in range(3)])
    return v


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    with torch.no_grad():
        if kind == "batch":
            return [_filter(a, _spectrum(p, a.shape)) for a, p in zip(s["images"], s["psfs"])]
        if kind == "rl":
            views = [v.double() for v in s["views"]]
            spectra = [_spectrum(p, views[0].shape) for p in s["psfs"]]
            psi = sum(views) / len(views)
            for _ in range(s["iterations"]):
                total = 0
                for v, h in zip(views, spectra):
                    blur = _filter(psi, h).clamp_min_(float(np.float32(1e-6)))
                    total = total + _filter(v / blur, h, adjoint=True)
                psi = psi * (total / len(views))
            return psi
        if kind == "host":
            image = torch.from_numpy(s["image"].reshape(s["n"][::-1]))
            psf = torch.from_numpy(s["psf"].reshape(s["k"][::-1]))
            return _filter(image, _spectrum(psf, image.shape)).reshape(-1).numpy()
        image, psf = s["image"].detach(), s["psf"].detach()
        if kind == "boundary":
            wide = _extended(image, psf.shape, s["mode"])
            out = _filter(wide, _spectrum(psf, wide.shape))
            z, y, x = (k - 1 - k // 2 for k in psf.shape)
            nz, ny, nx = image.shape
            return out[z:z + nz, y:y + ny, x:x + nx].contiguous()
        h = _spectrum(psf, image.shape)
        if kind != "train":
            return _filter(image, h, adjoint=kind == "correlate")
        lag = torch.fft.irfftn(torch.fft.rfftn(s["grad"].double()) *
                               torch.fft.rfftn(image.double()).conj(), s=image.shape)
        z, y, x = ((torch.arange(k, device=psf.device) - k // 2) % n
                   for k, n in zip(psf.shape, image.shape))
        return {"out": _filter(image, h), "grad_image": _filter(s["grad"], h, adjoint=True),
                "grad_psf": lag[z[:, None, None], y[None, :, None], x[None, None, :]]}
