"""Graph capture of calls on extended axes whose lengths have no tables yet
(the file's name puts it before the tests that use every length).  The
captured calls then run the image's own lengths; every replay is checked,
with eager work and synchronisation between replays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5  # as in test_gpu_extension.py


def test_capture_with_a_kernel_size_not_seen(fc, oracle):
    import torch
    from fourierconvolutioncudalib_amd import synth
    from fourierconvolutioncudalib_amd.autograd import grad_kernel
    shape, small, large = (36, 190, 254), (3, 3, 3), (5, 12, 40)  # x 256, then 300; y 192, 210
    k0 = torch.from_numpy(synth.random_psf(small, 1)).cuda()
    k = torch.from_numpy(synth.random_psf(large, 2)).cuda()
    data = [torch.from_numpy(synth.uniform(shape, 10 + i)).cuda() for i in range(3)]
    g0 = torch.from_numpy(np.random.default_rng(3).standard_normal(shape).astype(np.float32)).cuda()
    src = data[0].clone()
    out, planned = torch.empty_like(src), torch.empty_like(src)
    ws = torch.empty(fc.workspace_bytes(shape, large), dtype=torch.uint8, device="cuda")
    pws = torch.empty_like(ws)
    # the lengths that the small kernel's extension needs are there; the one
    # eager call of the image's extents is with that kernel
    fc.convolve3d(torch.rand(36, 192, 256, device="cuda"), k0)
    fc.convolve3d(src, k0)
    torch.cuda.synchronize()
    graph, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    print("capture", shape, large, flush=True)
    with torch.cuda.stream(s):
        with torch.cuda.graph(graph, stream=s):
            fc.convolve3d(src, k, out=out, workspace=ws, stream=s)
            plan = fc.ConvolutionPlan(shape, k, workspace=pws, stream=s)
            plan.run(src, out=planned, stream=s)
            dk = grad_kernel(g0, src, large, stream=s)
    for d in data:
        src.copy_(d)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        a, n = d.cpu().numpy(), k.cpu().numpy()
        ref = oracle.numpy_fft_conv(a, n)
        assert oracle.rel_l2(out.cpu().numpy(), ref) < TOL
        assert oracle.rel_l2(planned.cpu().numpy(), ref) < TOL
        want = oracle.fft_conv_grad_kernel(g0.cpu().numpy(), a, large)
        assert oracle.rel_l2(dk.cpu().numpy(), want) < TOL
        src.mul_(0.5)
        out.zero_()
        torch.cuda.synchronize()
    plan.close()
    # eager afterwards, on the extended lengths
    fc.convolve3d(data[0], k, out=out)
    ref = oracle.numpy_fft_conv(data[0].cpu().numpy(), k.cpu().numpy())
    assert oracle.rel_l2(out.cpu().numpy(), ref) < TOL
