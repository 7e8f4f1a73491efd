"""Convolutions whose axes have no compile-time kernels run as extended
transforms (AxisExt in kernels.hpp): against the FP64 oracle at the extents
and kernel sizes where the extension can go wrong."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5

# image (z, y, x), kernel (z, y, x): one extended axis at a time and all
# three; odd extents (a lone last row of a plane, unaligned rows); kernels of
# one tap, even, and of the whole image; the last length before a compile-time
# one; whole-plane x and y kernels with an extended z; the largest registered
# transform length
SHAPES = [((64, 64, 67), (5, 5, 9)),
          ((64, 51, 64), (5, 8, 5)),
          ((65, 64, 128), (9, 3, 3)),
          ((61, 67, 71), (1, 1, 1)),
          ((61, 67, 71), (7, 4, 10)),
          ((31, 33, 47), (31, 33, 47)),
          ((127, 95, 63), (2, 2, 2)),
          ((49, 99, 251), (49, 15, 31)),
          ((36, 40, 3401), (3, 5, 95))]


def _data(shape, kshape, seed):
    from fourierconvolutioncudalib_amd import synth
    return synth.uniform(shape, seed), synth.random_psf(kshape, seed + 1)


@pytest.mark.parametrize("shape,kshape", SHAPES)
def test_extended_convolution(fc, oracle, shape, kshape):
    import torch
    a, k = _data(shape, kshape, 4100 + sum(shape))
    ta, tk = torch.from_numpy(a).cuda(), torch.from_numpy(k).cuda()
    for op, conj in ((fc.CONVOLVE, False), (fc.CORRELATE, True)):
        print("extended", shape, kshape, op, flush=True)
        ref = oracle.numpy_fft_conv(a, k, conj_kernel=conj)
        got = fc.convolve3d(ta, tk, op=op)
        assert oracle.rel_l2(got.cpu().numpy(), ref) < TOL
        # a view that starts 4 bytes past an aligned address, in place
        buf = torch.empty(a.size + 1, device="cuda")
        off = buf[1:].view(a.shape).copy_(ta)
        fc.convolve3d(off, tk, op=op, out=off)
        assert torch.equal(off, got)
    # the host entry point
    assert oracle.rel_l2(fc.convolve(a, k), oracle.numpy_fft_conv(a, k)) < TOL


@pytest.mark.parametrize("mode", ["zero", "nearest", "reflect", "mirror"])
@pytest.mark.parametrize("shape,kshape", [((40, 48, 61), (15, 4, 31)),
                                          # the reach of one fold: 32 and 33 elements past an end
                                          ((33, 40, 48), (67, 1, 3)),
                                          ((33, 40, 48), (68, 3, 1))])
def test_extended_boundary(fc, oracle, mode, shape, kshape):
    import torch
    a, k = _data(shape, kshape, 4300 + sum(kshape))
    ta, tk = torch.from_numpy(a).cuda(), torch.from_numpy(k).cuda()
    for op in (fc.CONVOLVE, fc.CORRELATE):
        print("boundary", mode, shape, kshape, op, flush=True)
        got = fc.convolve3d_boundary(ta, tk, mode, op=op).cpu().numpy()
        ref = oracle.boundary_conv_direct(a, k, mode, correlate=op == fc.CORRELATE)
        assert oracle.rel_l2(got, ref) < TOL


def test_unextended_workspace_is_enough(fc, oracle):
    """A workspace that holds the plain transform serves the call too."""
    import torch
    from fourierconvolutioncudalib_amd._lib import check, ints
    a, k = _data((61, 67, 71), (7, 4, 10), 4500)
    ta, tk = torch.from_numpy(a).cuda(), torch.from_numpy(k).cuda()
    fc.use_static_kernels(False)
    small = fc.workspace_bytes(a.shape, k.shape)
    fc.use_static_kernels(True)
    assert small < fc.workspace_bytes(a.shape, k.shape)
    ws = torch.empty(small, dtype=torch.uint8, device="cuda")
    out = torch.empty_like(ta)
    check(fc.lib().fcamd_convolve3d_device(out.data_ptr(), ta.data_ptr(), ints(a.shape[::-1]),
                                           tk.data_ptr(), ints(k.shape[::-1]), fc.CONVOLVE,
                                           ws.data_ptr(), small, None))
    torch.cuda.synchronize()
    assert oracle.rel_l2(out.cpu().numpy(), oracle.numpy_fft_conv(a, k)) < TOL


@pytest.mark.parametrize("shape,kshape", [((64, 64, 67), (5, 5, 9)), ((61, 51, 64), (61, 8, 5)),
                                          ((61, 67, 71), (7, 4, 10)), ((37, 33, 47), (37, 33, 47)),
                                          ((300, 33, 41), (31, 1, 2))])
def test_extended_gradients(fc, oracle, shape, kshape):
    """Both gradients of extended shapes through torch autograd."""
    import torch
    from fourierconvolutioncudalib_amd.autograd import fft_conv3d
    a, k = _data(shape, kshape, 4700 + sum(shape))
    g = np.random.default_rng(4701).standard_normal(shape).astype(np.float32)
    ta = torch.from_numpy(a).cuda().requires_grad_(True)
    tk = torch.from_numpy(k).cuda().requires_grad_(True)
    print("gradients", shape, kshape, flush=True)
    fft_conv3d(ta, tk).backward(torch.from_numpy(g).cuda())
    assert oracle.rel_l2(ta.grad.cpu().numpy(), oracle.numpy_fft_conv(g, k, conj_kernel=True)) < TOL
    assert oracle.rel_l2(tk.grad.cpu().numpy(), oracle.fft_conv_grad_kernel(g, a, kshape)) < TOL
