"""How the library would run a convolution, asked on the CPU: a small program
(tests/routes/routes.cpp) linked against the static archive prints a problem's
transform lengths, whether it takes the whole-plane kernels, and its
workspace."""
import math
import os
import random
import subprocess

import pytest

from test_gpu_planes import REGULAR_PLANES, WIDE_PLANES

ROOT = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..")
MODES = {"periodic": 0, "zero": 1, "nearest": 2, "reflect": 3, "mirror": 4}


def _build(fc, directory, name, *link):
    prog = str(directory / name)
    archive = os.path.join(os.path.dirname(fc._lib.LIB_PATH),
                           "libFourierConvolutionCUDALib_static.a")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", fc._lib.CSRC,
                    "-I/opt/rocm/include", os.path.join(ROOT, "tests", "routes", name + ".cpp"),
                    archive, "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib",
                    "-lpthread", *link, "-o", prog], check=True)
    return prog


@pytest.fixture(scope="session")
def routes(fc, tmp_path_factory):
    """routes([(nx, ny, nz, kx, ky, kz, boundary), ...]) -> [(px, py, pz,
    plane forward, plane inverse, workspace bytes), ...]"""
    prog = _build(fc, tmp_path_factory.mktemp("routes"), "routes")

    def ask(problems):
        # every split form on, so that no rule asks a device for its CU count
        env = dict(os.environ, FCAMD_PLANE_SPLIT="1")
        env.pop("FCAMD_NO_PLANES", None)
        env.pop("FCAMD_NO_STATIC", None)
        r = subprocess.run([prog], input="\n".join(" ".join(map(str, p)) for p in problems),
                           env=env, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        out = [tuple(int(v) for v in line.split()) for line in r.stdout.splitlines()]
        assert len(out) == len(problems)
        return out

    return ask


def test_extended_planes_take_no_plane_kernel(routes):
    """Every plane extent with whole-plane kernels, in every boundary mode: a
    transform longer than the plane in x or y has no such kernel (they run the
    image's own plane as a circular one); a plane of its own extents has."""
    planes = REGULAR_PLANES + WIDE_PLANES
    problems = [(nx, ny, 64, kx, ky, kz, b) for nx, ny in planes
                for kx, ky, kz in ((9, 9, 9), (3, 1, 1), (1, 3, 1), (1, 1, 9), (1, 1, 1))
                for b in MODES.values()]
    extended = plain = 0
    for p, (px, py, _, fwd, inv, _) in zip(problems, routes(problems)):
        if (px, py) != p[:2]:
            assert (fwd, inv) == (0, 0), p
            extended += 1
        else:
            assert fwd or inv, p
            plain += 1
    # longer in x or y: 3 kernels x 4 modes of every plane
    assert extended == 12 * len(planes) and plain == 13 * len(planes)


# (image, kernel) x y z, and whether its axes are extended: the two sides of
# each line of extension_pays (conv_driver.cpp)
EXTENDED = [((509, 1, 500), (9, 1, 9), False), ((509, 1, 128), (3, 1, 5), True),
            ((509, 3, 500), (9, 3, 9), True), ((3001, 1, 2000), (5, 1, 3), False),
            ((3001, 2, 512), (5, 1, 3), False), ((1, 509, 2000), (1, 5, 3), True),
            ((1, 1511, 2000), (1, 5, 3), False),
            ((64, 64, 1), (3, 3, 1), False), ((126, 126, 1), (9, 9, 1), True),
            ((252, 252, 128), (101, 101, 128), True), ((252, 252, 128), (252, 252, 128), False),
            ((13, 14, 512), (3, 3, 3), False), ((22, 5, 512), (3, 1, 5), False),
            ((31, 31, 31), (31, 31, 31), True), ((143, 5, 512), (5, 1, 3), True),
            ((14, 512, 64), (3, 3, 3), False), ((36, 512, 64), (18, 18, 18), False),
            ((252, 512, 64), (3, 3, 3), True), ((20, 512, 90), (3, 3, 3), True),
            ((50, 64, 64), (15, 11, 39), True), ((126, 448, 70), (31, 31, 33), True),
            ((128, 128, 21), (3, 3, 10), True), ((126, 240, 48), (13, 39, 31), True),
            ((19, 384, 35), (1, 32, 3), False),
            ((13, 512, 64), (3, 3, 3), False), ((104, 512, 64), (52, 52, 52), True),
            ((17, 512, 64), (3, 3, 3), False), ((23, 64, 64), (3, 3, 3), True),
            ((158, 158, 218), (31, 31, 91), True), ((286, 286, 346), (31, 31, 91), True)]


def test_where_an_extension_pays(routes):
    got = routes([(*n, *k, 0) for n, k, _ in EXTENDED])
    for (n, k, want), g in zip(EXTENDED, got):
        assert (g[:3] != n) == want, (n, k, g)


EXTENDED_GRADIENTS = [((128, 28, 128), (14, 14, 14), False), ((256, 63, 256), (3, 3, 3), True),
                      ((126, 126, 126), (6, 6, 6), True), ((14, 22, 512), (3, 3, 3), False),
                      ((256, 26, 256), (3, 3, 3), True), ((17, 20, 512), (3, 3, 3), False),
                      ((64, 23, 64), (3, 3, 3), True), ((36, 512, 64), (18, 18, 18), False),
                      ((64, 64, 14), (3, 3, 3), False), ((256, 256, 168), (3, 3, 3), True),
                      ((55, 512, 14), (27, 27, 14), False), ((64, 64, 13), (3, 3, 3), False),
                      ((77, 512, 64), (3, 3, 3), True), ((17, 512, 64), (3, 3, 3), False),
                      ((23, 64, 64), (3, 3, 3), False), ((58, 512, 64), (3, 3, 3), True),
                      ((75, 54, 48), (25, 11, 19), True), ((23, 248, 130), (23, 189, 94), True),
                      ((26, 29, 133), (9, 11, 49), True), ((88, 100, 195), (35, 17, 7), True),
                      ((158, 158, 218), (31, 31, 91), True), ((509, 1, 500), (9, 1, 9), False)]


def test_where_an_extended_gradient_pays(routes):
    got = routes([(*n, *k, 5) for n, k, _ in EXTENDED_GRADIENTS])
    for (n, k, want), g in zip(EXTENDED_GRADIENTS, got):
        assert (g[:3] != n) == want, (n, k, g)


def test_extended_workspace_is_bounded(routes, fc):
    """Past 32 MiB no convolution asks for more than 13 times the workspace
    of its own extents."""
    rng = random.Random(7)
    problems = []
    while len(problems) < 3000:
        n = [int(round(math.exp(rng.uniform(0, math.log(3413))))) for _ in range(3)]
        if n[0] * n[1] * n[2] > 1 << 28:
            continue
        f = rng.choice([0.03, 0.3, 1.0])
        problems.append((*n, *(max(1, int(f * d * rng.uniform(0.5, 1.0))) for d in n), 0))
    fc.use_static_kernels(False)
    try:
        plain = [fc.workspace_bytes(p[2::-1], p[5:2:-1]) for p in problems]
    finally:
        fc.use_static_kernels(True)
    for p, own, got in zip(problems, plain, routes(problems)):
        assert got[5] <= max(32 << 20, 13 * own), (p, own, got)


def test_workspace_where_memory_ends(fc, tmp_path):
    """The pool's workspace for an extended transform, or for the unextended
    one where the device has no memory for that; an error where it has for
    neither."""
    prog = _build(fc, tmp_path, "reserve", "-Wl,--wrap=hipMalloc,--wrap=hipFree,"
                  "--wrap=hipDeviceSynchronize")
    # memory, already held, wanted, enough -> returned, held afterwards, last request
    cases = {(1000, 0, 800, 300): "800 800 800", (1000, 900, 800, 300): "800 900 0",
             (500, 0, 800, 300): "300 300 300", (500, 400, 800, 300): "300 300 300",
             (200, 0, 800, 300): "error 3 0", (500, 0, 800, 800): "error 3 0"}
    r = subprocess.run([prog], input="\n".join(" ".join(map(str, c)) for c in cases),
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    assert r.stdout.splitlines() == list(cases.values())


def test_tensor_workspace_where_memory_ends(fc, monkeypatch):
    """Without memory for a call's workspace the wrapper leaves it to the
    library."""
    import torch

    def empty(*a, **k):
        raise torch.OutOfMemoryError("no memory")

    monkeypatch.setattr(torch, "empty", empty)
    assert fc._workspace(1 << 20, None, torch.device("cpu"), None) == (None, 0, None)


_DEVICE_CALLS = ("hipMalloc", "hipFree", "hipMemcpy", "hipGetDevice", "hipGetLastError",
                 "hipStreamIsCapturing", "__hipPushCallConfiguration",
                 "__hipPopCallConfiguration", "hipLaunchKernel", "hipFuncSetAttribute",
                 "hipDeviceGetAttribute", "hipOccupancyMaxActiveBlocksPerMultiprocessor",
                 "hipStreamCreateWithFlags", "hipStreamDestroy", "hipEventCreateWithFlags",
                 "hipEventDestroy")


@pytest.fixture(scope="session")
def steps(fc, tmp_path_factory):
    """steps([(what, capturing, image, kernel), ...]) -> per step (launches,
    allocations), or the status code of a refusal (tests/routes/capture.cpp);
    every call starts from a process without tables"""
    prog = _build(fc, tmp_path_factory.mktemp("capture"), "capture",
                  "-Wl," + ",".join("--wrap=" + c for c in _DEVICE_CALLS))
    env = {k: v for k, v in os.environ.items() if not k.startswith("FCAMD_")}

    def run(what):
        r = subprocess.run([prog], input="\n".join(" ".join(map(str, (w, c, *n, *k)))
                                                   for w, c, n, k in what),
                           env=env, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        out = [line.split() for line in r.stdout.splitlines()]
        assert len(out) == len(what)
        return [int(o[1]) if o[0] == "error" else tuple(map(int, o)) for o in out]

    return run


CONV, GRADIENT, PLAN, BATCH = range(4)


@pytest.mark.parametrize("first", [CONV, GRADIENT, PLAN, BATCH])
@pytest.mark.parametrize("then", [CONV, GRADIENT, PLAN])
def test_capture_after_any_kernel_size(steps, first, then):
    """One eager call of an image's extents is enough to capture calls of any
    kernel size on it, also where the first call's extended lengths were
    there already and the second's are not."""
    n = (126, 126, 126)  # extends to 128 with 3 taps, to 144 with 13
    got = steps([(CONV, 0, (128, 128, 128), (3, 3, 3)), (first, 0, n, (3, 3, 3)),
                 (then, 1, n, (13, 13, 13)), (then, 0, n, (13, 13, 13)),
                 (then, 1, n, (13, 13, 13))])
    assert got[1][1] > 0, "no table of the image's own extents"
    assert got[2][0] > 0 and got[2][1] == 0, "captured"
    assert got[3][0] > 0 and got[4][0] > 0 and got[4][1] == 0


def test_capture_without_any_call_is_refused(steps):
    n, k = (126, 126, 126), (3, 3, 3)
    assert steps([(CONV, 1, n, k), (GRADIENT, 1, n, k)]) == [1, 1]
    # and what is captured with its tables there allocates nothing
    assert steps([(CONV, 0, n, k), (CONV, 1, n, k)])[1][1] == 0


def test_current_stream_without_the_raw_handle(fc, monkeypatch):
    """The current stream's handle from torch's public interface where the
    direct one is not there."""
    import torch

    class Stream:
        cuda_stream = 4096

    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: Stream())
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    assert fc._stream_handle(None).value == 4096
