"""Calls on extended axes whose workspace, table or budget only holds the
unextended transform."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# as in test_gpu_extension.py; Richardson-Lucy as in test_gpu_rl.py
TOL, RL_TOL = 1e-5, 1e-4
SHAPE, KSHAPE = (61, 67, 71), (7, 4, 10)  # every axis is extended


def _plain(fc, f):
    """f() with the compile-time kernels off, so that no axis is extended"""
    fc.use_static_kernels(False)
    try:
        return f()
    finally:
        fc.use_static_kernels(True)


def _data(seed):
    from fourierconvolutioncudalib_amd import synth
    return synth.uniform(SHAPE, seed), synth.random_psf(KSHAPE, seed + 1)


def test_rl_in_an_unextended_workspace(fc, oracle):
    import torch
    from fourierconvolutioncudalib_amd import synth
    from fourierconvolutioncudalib_amd._lib import check, ints
    _, views, psfs = synth.multiview((30, 29, 31), (7, 5, 9), 2, 77, sigma_xyz=(1.0, 1.0, 2.5),
                                     blobs_count=40)
    L = fc.lib()
    dims, kdims = ints((31, 29, 30)), ints((9, 5, 7) * 2)
    small = _plain(fc, lambda: L.fcamd_rl_workspace_bytes(2, dims, kdims, 1))
    assert 0 < small < L.fcamd_rl_workspace_bytes(2, dims, kdims, 1)
    tv = [torch.from_numpy(v).cuda() for v in views]
    tk = [torch.from_numpy(k).cuda() for k in psfs]
    vp = (ctypes.c_void_p * 2)(*[t.data_ptr() for t in tv])
    kp = (ctypes.c_void_p * 2)(*[t.data_ptr() for t in tk])
    psi = torch.empty_like(tv[0])
    ws = torch.empty(small, dtype=torch.uint8, device="cuda")
    print("Richardson-Lucy, unextended workspace", flush=True)
    check(L.fcamd_rl_multiview_device(psi.data_ptr(), vp, 2, dims, kp, kdims, 10, 1e-6, 1, 1,
                                      ws.data_ptr(), small, None))
    torch.cuda.synchronize()
    ref = oracle.rl_multiview(np.stack(views), psfs, 10, eps=1e-6)
    assert oracle.rel_l2(psi.cpu().numpy(), ref) < RL_TOL
    rc = L.fcamd_rl_multiview_device(psi.data_ptr(), vp, 2, dims, kp, kdims, 1, 1e-6, 1, 1,
                                     ws.data_ptr(), small - 256, None)
    assert rc == 1 and b"workspace" in L.fcamd_last_error_message()
