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


def test_unextended_workspace_of_tensor_calls(fc, oracle):
    """The tensor calls take a workspace of the unextended size and refuse
    less than that before any launch."""
    import torch
    from fourierconvolutioncudalib_amd.autograd import grad_kernel, grad_kernel_workspace_bytes
    a, k = _data(8100)
    g = np.random.default_rng(8101).standard_normal(SHAPE).astype(np.float32)
    ta, tk, tg = (torch.from_numpy(x).cuda() for x in (a, k, g))
    ref = oracle.numpy_fft_conv(a, k)
    dref = oracle.fft_conv_grad_kernel(g, a, KSHAPE)
    conv = fc.workspace_bytes(SHAPE, KSHAPE)
    small = _plain(fc, lambda: fc.workspace_bytes(SHAPE, KSHAPE))
    grad = grad_kernel_workspace_bytes(SHAPE, KSHAPE)
    gsmall = _plain(fc, lambda: grad_kernel_workspace_bytes(SHAPE, KSHAPE))
    assert 0 < small < conv and 0 < gsmall < grad

    def calls(n, gn):
        ws = torch.empty(n, dtype=torch.uint8, device="cuda")
        gws = torch.empty(gn, dtype=torch.uint8, device="cuda")
        yield "convolve3d", lambda: fc.convolve3d(ta, tk, workspace=ws), ref
        yield "periodic", lambda: fc.convolve3d_boundary(ta, tk, "periodic", workspace=ws), ref
        yield "plan", lambda: fc.ConvolutionPlan(SHAPE, tk, workspace=ws).run(ta), ref
        yield "gradient", lambda: grad_kernel(tg, ta, KSHAPE, workspace=gws), dref

    for name, call, want in calls(small, gsmall):
        print("unextended workspace", name, flush=True)
        assert oracle.rel_l2(call().cpu().numpy(), want) < TOL, name
    for n, gn in ((small - 256, gsmall - 256), (0, 0)):
        for name, call, _ in calls(n, gn):
            with pytest.raises(ValueError, match="workspace"):
                call()


def test_unextended_batch_workspace(fc, oracle, monkeypatch):
    import torch
    from fourierconvolutioncudalib_amd._lib import check, ints
    monkeypatch.setenv("FCAMD_BATCH_LANES", "2")
    L = fc.lib()
    a, k = _data(8200)
    b, q = _data(8210)
    ts = [torch.from_numpy(x).cuda() for x in (a, b)]
    ks = [torch.from_numpy(x).cuda() for x in (k, q)]
    outs = [torch.empty_like(t) for t in ts]
    dims, kdims = ints(SHAPE[::-1] * 2), ints(KSHAPE[::-1] * 2)
    need = L.fcamd_batch_workspace_bytes(2, dims, kdims)
    small = _plain(fc, lambda: L.fcamd_batch_workspace_bytes(2, dims, kdims))
    assert 0 < small < need
    ws = torch.empty(small, dtype=torch.uint8, device="cuda")
    ptrs = lambda x: (ctypes.c_void_p * 2)(*[t.data_ptr() for t in x])  # noqa: E731
    print("unextended batch workspace", flush=True)
    plan = L.fcamd_batch_create(2, dims, kdims, ptrs(outs), ptrs(ts), ptrs(ks), fc.CONVOLVE,
                                ws.data_ptr(), small)
    assert plan
    check(L.fcamd_batch_execute(plan, None))
    torch.cuda.synchronize()
    L.fcamd_batch_destroy(plan)
    for o, x, y in zip(outs, (a, b), (k, q)):
        assert oracle.rel_l2(o.cpu().numpy(), oracle.numpy_fft_conv(x, y)) < TOL
    assert not L.fcamd_batch_create(2, dims, kdims, ptrs(outs), ptrs(ts), ptrs(ks), fc.CONVOLVE,
                                    ws.data_ptr(), small - 256)


def test_host_budget_between_the_sizes(fc, oracle, monkeypatch):
    """A device budget that holds the unextended single shot only."""
    from fourierconvolutioncudalib_amd._lib import ints
    shape, kshape = (61, 135, 142), (9, 9, 91)  # x grows from 142 to 240
    from fourierconvolutioncudalib_amd import synth
    a, k = synth.uniform(shape, 8300), synth.random_psf(kshape, 8301)
    L = fc.lib()

    def need():
        return L.fcamd_host_device_bytes(ints(shape[::-1]), ints(kshape[::-1]), 0)

    monkeypatch.setenv("FCAMD_DEVICE_BUDGET_MB", "4096")
    large, small = need(), _plain(fc, need)
    budget = -(-small >> 20)
    assert small <= budget << 20 < large
    monkeypatch.setenv("FCAMD_DEVICE_BUDGET_MB", str(budget))
    assert need() <= budget << 20
    print("host budget", budget, "MiB of", large >> 20, flush=True)
    assert oracle.rel_l2(fc.convolve(a, k), oracle.numpy_fft_conv(a, k)) < TOL
