"""Fused SwiGLU (naylis_mom_swiglu_*) against transformers' LlamaMLP
activation, silu(gate) * up, on the same GPU inputs (model.py:279-345)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(16384, 2816), (3, 7, 64), (8,)])
def test_swiglu_matches_silu_times_up(shape, dtype, dev):
    from naylis_amd.mom_kernels.hip_mlp import swiglu
    g0 = torch.Generator().manual_seed(sum(shape))
    g = (torch.randn(shape, generator=g0) * 3).to(dtype).to(dev)
    u = torch.randn(shape, generator=g0).to(dtype).to(dev)
    dh = torch.randn(shape, generator=g0).to(dtype).to(dev)
    gr, ur = g.clone().requires_grad_(True), u.clone().requires_grad_(True)
    hr = F.silu(gr) * ur
    hr.backward(dh)
    gg, ug = g.clone().requires_grad_(True), u.clone().requires_grad_(True)
    hg = swiglu(gg, ug)
    hg.backward(dh)
    torch.cuda.synchronize()
    if dtype == torch.bfloat16:
        # the same bf16 roundings; silu's fp32 value may differ in its last bit
        # from torch's (separately compiled exp / division), which can move a
        # bf16 rounding by one ulp
        for got, want in ((hg, hr), (gg.grad, gr.grad), (ug.grad, ur.grad)):
            ulp2 = (want.float().abs() * 2.0 ** -6).clamp_min(1e-30)
            assert bool(((got.float() - want.float()).abs() <= ulp2).all())
            assert float((got != want).float().mean()) < 1e-3
    else:
        assert torch.allclose(hg, hr, rtol=1e-6, atol=1e-7)
        assert torch.allclose(gg.grad, gr.grad, rtol=1e-5, atol=1e-6)
        assert torch.allclose(ug.grad, ur.grad, rtol=1e-6, atol=1e-7)


def test_swiglu_rejects_unsupported(dev):
    from naylis_amd.mom_kernels.hip_mlp import swiglu
    with pytest.raises(RuntimeError, match="unsupported"):
        swiglu(torch.randn(7, device=dev), torch.randn(7, device=dev))


def test_status_error_in_a_backward_keeps_its_type(dev):
    """A C-ABI call that refuses its arguments inside a backward (here a gradient
    at an odd address) raises NaylisError with its code, as in a forward."""
    from naylis_amd import _lib
    from naylis_amd.mom_kernels.hip_mlp import swiglu
    g, u = (torch.randn(4, 64, device=dev).bfloat16().requires_grad_() for _ in range(2))
    buf = torch.zeros(4 * 64 + 1, device=dev).bfloat16()
    h = swiglu(g, u)
    with pytest.raises(_lib.NaylisError) as err:
        h.backward(buf[1:].view(4, 64))
    assert err.value.code == _lib.NAYLIS_ERR_ARG and "aligned" in str(err.value)
    with pytest.raises(_lib.NaylisError) as err, torch.no_grad():
        swiglu(buf[1:].view(4, 64), u)
    assert err.value.code == _lib.NAYLIS_ERR_ARG


def test_backward_launches_on_the_current_stream(dev):
    """A backward called directly on another stream than the forward's launches
    there: under capture its kernel is in the graph, and replays follow their
    inputs."""
    from naylis_amd.mom_kernels.hip_mlp import swiglu
    gen = torch.Generator(device=dev).manual_seed(3)
    g, u = (torch.randn(64, 64, generator=gen, device=dev).bfloat16().requires_grad_() for _ in range(2))
    dys = [torch.randn(64, 64, generator=gen, device=dev).bfloat16() for _ in range(3)]
    h = swiglu(g, u)
    want = [torch.autograd.grad(h, (g, u), d, retain_graph=True) for d in dys]
    dy = dys[0].clone()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        got = h.grad_fn(dy)
    for d, w in zip(dys, want):
        dy.copy_(d)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got[0], w[0]) and torch.equal(got[1], w[1])
