"""Boundary-mode convolutions of images whose plane has whole-plane kernels
for its circular transform: the boundary's longer transform must not take
them.  Against the FP64 FFT oracle, through the device and the host entry
point."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# as in test_gpu_boundary.py
TOL = 1e-5

# (image, kernel) in C order: one-workgroup planes, wide planes that split in
# one or both directions, an inverse-only wide plane (240 x 240), a kernel
# that leaves x or y alone
CASES = [((33, 64, 64), (5, 5, 5)),
         ((64, 128, 128), (15, 15, 15)),
         ((40, 256, 64), (3, 9, 7)),
         ((64, 64, 192), (7, 4, 11)),
         ((32, 192, 192), (5, 9, 9)),
         ((40, 240, 240), (3, 5, 5)),
         ((128, 256, 256), (9, 15, 15)),
         ((20, 64, 64), (3, 1, 5)),
         ((20, 64, 64), (3, 5, 1)),
         ((20, 64, 64), (7, 1, 1))]


@pytest.mark.parametrize("mode", ["zero", "nearest", "reflect", "mirror"])
@pytest.mark.parametrize("shape,kshape", CASES)
def test_boundary_on_plane_extents(fc, oracle, shape, kshape, mode):
    import torch
    from fourierconvolutioncudalib_amd import synth
    from fourierconvolutioncudalib_amd._lib import check, ints
    a = synth.uniform(shape, 6100 + sum(shape))
    k = synth.random_psf(kshape, 6200 + sum(kshape))
    ta, tk = torch.from_numpy(a).cuda(), torch.from_numpy(k).cuda()
    fp = ctypes.POINTER(ctypes.c_float)
    for op in (fc.CONVOLVE, fc.CORRELATE):
        print("boundary plane", mode, shape, kshape, op, flush=True)
        ref = oracle.fft_boundary_conv(a, k, mode, correlate=op == fc.CORRELATE)
        got = fc.convolve3d_boundary(ta, tk, mode, op=op).cpu().numpy()
        assert oracle.rel_l2(got, ref) < TOL
        im = np.ascontiguousarray(a.copy())
        check(fc.lib().fcamd_convolve3d_boundary_host(
            im.ctypes.data_as(fp), ints(shape[::-1]), k.ctypes.data_as(fp), ints(kshape[::-1]),
            op, fc.BOUNDARY[mode], 0))
        assert oracle.rel_l2(im, ref) < TOL
