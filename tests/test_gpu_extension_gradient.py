"""PSF gradients on extended axes (conv_driver.cpp): the kernel's rows taken
directly or through the x pass, at the line between the two."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# as in test_gpu_extension.py
TOL = 1e-5


def _x_inverses(fc, f):
    """Runs f and returns how many x inverse passes it launched."""
    L = fc.lib()
    ms, counts = (ctypes.c_double * 16)(), (ctypes.c_int * 16)()
    L.fcamd_pass_timing(1)
    try:
        f()
    finally:
        L.fcamd_pass_timing(0)
    n = L.fcamd_pass_times(ms, counts, 16)
    return sum(counts[i] for i in range(n) if L.fcamd_pass_name(i) == b"image_xinv")


# y extends to 80 rows: 34 * 37 taps are within 16 of them, 35 * 37 are not;
# a registered y; an odd lone plane; the whole image
@pytest.mark.parametrize("shape,kshape,rows", [((20, 37, 61), (7, 37, 34), 0),
                                               ((20, 37, 61), (7, 37, 35), 1),
                                               ((33, 64, 67), (5, 64, 17), 1),
                                               ((33, 64, 67), (1, 64, 16), 0),
                                               ((41, 53, 67), (41, 53, 67), 1)])
def test_rows_of_large_kernels(fc, oracle, shape, kshape, rows):
    import torch
    from fourierconvolutioncudalib_amd import synth
    from fourierconvolutioncudalib_amd.autograd import grad_kernel
    a = synth.uniform(shape, 7100 + sum(shape))
    g = np.random.default_rng(7101).standard_normal(shape).astype(np.float32)
    ta, tg = torch.from_numpy(a).cuda(), torch.from_numpy(g).cuda()
    print("gradient rows", shape, kshape, flush=True)
    got = []
    assert _x_inverses(fc, lambda: got.append(grad_kernel(tg, ta, kshape))) == rows
    assert oracle.rel_l2(got[0].cpu().numpy(), oracle.fft_conv_grad_kernel(g, a, kshape)) < TOL
