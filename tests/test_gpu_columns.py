"""z transforms with two-stage plans and with kernel columns cut to the slots
their taps reach, and x transforms of partly filled workgroups, against the
FP64 oracle at the sizes where those rules change over."""
import pytest

pytestmark = pytest.mark.gpu

# five passes, each a chain of at most log2(n) butterfly levels of three
# roundings (unit roundoff 6e-8): 3 * 6e-8 * 2 * log2(64 * 64 * 432) = 7.5e-6
TOL = 1e-5


@pytest.mark.parametrize("nz", [64, 96, 105, 128, 160, 192, 200, 216, 224, 256, 270, 288, 300,
                                336, 384, 400, 432, 512])
def test_kernel_columns(fc, oracle, nz):
    """Taps around a quarter and a half of the column (and what a quarter is
    rounded up to in whole slots), whole columns, one tap."""
    import torch
    from fourierconvolutioncudalib_amd import synth
    a = synth.uniform((nz, 64, 64), 5100 + nz)
    ta = torch.from_numpy(a).cuda()
    for kz in sorted({1, 2, nz // 4 - 1, nz // 4, nz // 4 + 1, 3 * nz // 10, 3 * nz // 10 + 1,
                      nz // 3, nz // 2 - 1, nz // 2, nz // 2 + 1, 3 * nz // 5, 3 * nz // 5 + 1,
                      nz}):
        k = synth.random_psf((kz, 3, 2), 5200 + kz)
        tk = torch.from_numpy(k).cuda()
        for op, conj in ((fc.CONVOLVE, False), (fc.CORRELATE, True)):
            print("columns", nz, kz, op, flush=True)
            ref = oracle.numpy_fft_conv(a, k, conj_kernel=conj)
            got = fc.convolve3d(ta, tk, op=op)
            assert oracle.rel_l2(got.cpu().numpy(), ref) < TOL, kz


@pytest.mark.parametrize("rows", [(1, 1), (5, 5), (7, 6)])
def test_x_workgroups(fc, oracle, rows):
    """Every compile-time length over rows that fill no workgroup, leave a
    lone last row, and leave a partly filled last workgroup."""
    import torch
    from fourierconvolutioncudalib_amd import synth
    for nx in fc.static_lengths():
        a = synth.uniform((*rows, nx), 5300 + nx)
        k = synth.random_psf((1, min(rows[1], 3), 5), 5400 + nx)
        print("rows", rows, nx, flush=True)
        ref = oracle.numpy_fft_conv(a, k)
        got = fc.convolve3d(torch.from_numpy(a).cuda(), torch.from_numpy(k).cuda())
        assert oracle.rel_l2(got.cpu().numpy(), ref) < TOL, nx


@pytest.mark.parametrize("nz", [200, 216, 250, 270, 400])
def test_whole_second_columns(fc, oracle, nz):
    """PSF gradients and kernels past half the column, on lengths whose whole
    columns and cut ones run different plans (200, 250) and the same."""
    import numpy as np
    import torch
    from fourierconvolutioncudalib_amd import synth
    from fourierconvolutioncudalib_amd.autograd import grad_kernel
    shape = (nz, 33, 64)
    a = synth.uniform(shape, 5500 + nz)
    g = np.random.default_rng(5501).standard_normal(shape).astype(np.float32)
    ta, tg = torch.from_numpy(a).cuda(), torch.from_numpy(g).cuda()
    for kz in (1, 9, nz // 2 + 1, nz):
        kshape = (kz, 3, 5)
        print("whole columns", nz, kz, flush=True)
        got = grad_kernel(tg, ta, kshape).cpu().numpy()
        assert oracle.rel_l2(got, oracle.fft_conv_grad_kernel(g, a, kshape)) < TOL, kz
        k = synth.random_psf(kshape, 5600 + kz)
        got = fc.convolve3d(ta, torch.from_numpy(k).cuda()).cpu().numpy()
        assert oracle.rel_l2(got, oracle.numpy_fft_conv(a, k)) < TOL, kz
