"""Causal attention kernels (naylis_mom_attn_*) against fp64 attention on the
same bf16 inputs: sequence lengths around the tiles (32-row products, 64-row
stages, 128-row workgroups), one head and many."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [(1, 1, 1), (2, 31, 1), (1, 33, 3), (1, 64, 2), (2, 65, 2), (1, 127, 4), (1, 129, 1), (2, 257, 3),
         (1, 1021, 16), (24, 700, 8), (64, 257, 8), (3, 2048, 32)]


def _reference(q, k, v, scale, dout):
    """fp64 attention per head with its gradients and, for each result, the
    largest error that bf16 P / dS and one bf16 rounding of the result allow:
    a bf16 rounding is at most 2^-8 relative (half of the 2^-7 spacing at 1), so
    two are 2^-7 of the sum of the terms' magnitudes, plus the fp32 exponent's
    2^-16."""
    q, k, v, dout = (t.double().transpose(1, 2) for t in (q, k, v, dout))
    S = q.shape[2]
    s = q @ k.transpose(-1, -2) * scale
    s.masked_fill_(torch.ones(S, S, dtype=torch.bool, device=q.device).triu(1), -math.inf)
    p = torch.softmax(s, -1)
    o = p @ v
    dp = dout @ v.transpose(-1, -2)
    delta = (dout * o).sum(-1, keepdim=True)
    ds = p * (dp - delta) * scale
    # |dS|'s own error: P and o rounded to bf16 inside delta
    ads = p * (dp.abs() + delta.abs() + (dout.abs() * o.abs()).sum(-1, keepdim=True)) * scale
    pt, dst, adst = p.transpose(-1, -2), ds.transpose(-1, -2), ads.transpose(-1, -2)
    res = {"o": (o, p @ v.abs()), "dq": (ds @ k, ads @ k.abs()), "dk": (dst @ q, adst @ q.abs()),
           "dv": (pt @ dout, pt @ dout.abs())}
    return {n: (a.transpose(1, 2), b.transpose(1, 2) * (2.0 ** -7 + 2.0 ** -16)) for n, (a, b) in res.items()}


@pytest.mark.parametrize("B,S,H", CASES)
def test_attention_matches_fp64(B, S, H, dev):
    from naylis_amd.mom_kernels.hip_attention import causal_attention
    g = torch.Generator(device=dev).manual_seed(S)
    q, k, v, dout = (torch.randn(B, S, H, 64, generator=g, device=dev).bfloat16() for _ in range(4))
    q[:, S // 2:] *= 6  # sharp rows: the running reference has to move
    q, k, v = (t.requires_grad_() for t in (q, k, v))
    o = causal_attention(q, k, v, 0.125)
    o.backward(dout)
    with torch.no_grad():
        for b in range(B):  # one sequence at a time bounds the fp64 scores
            ref = _reference(q[b:b + 1], k[b:b + 1], v[b:b + 1], 0.125, dout[b:b + 1])
            got = {"o": o[b:b + 1], "dq": q.grad[b:b + 1], "dk": k.grad[b:b + 1], "dv": v.grad[b:b + 1]}
            for n, (want, bound) in ref.items():
                err = (got[n].double() - want).abs()
                assert bool((err <= bound + 1e-30).all()), (n, b, float((err / (bound + 1e-30)).max()))


def test_attention_is_deterministic_and_causal(dev):
    from naylis_amd.mom_kernels.hip_attention import causal_attention
    g = torch.Generator(device=dev).manual_seed(1)
    x = [torch.randn(2, 333, 4, 64, generator=g, device=dev).bfloat16() for _ in range(4)]

    def run(q, k, v, d):
        q, k, v = (t.clone().requires_grad_() for t in (q, k, v))
        o = causal_attention(q, k, v, 0.125)
        o.backward(d)
        return [o.detach(), q.grad, k.grad, v.grad]

    a, b = run(*x), run(*x)
    assert all(torch.equal(s, t) for s, t in zip(a, b))
    y = [t.clone() for t in x]
    for t in y[:3]:
        t[:, 200:] *= 7     # the future reaches no earlier output, bit for bit
    assert torch.equal(run(*y)[0][:, :200], a[0][:, :200])


def test_attention_module_route(dev):
    """NaylisAttention takes the kernels for plain causal bf16 attention and the
    configured backend with a mask or another head size; both agree."""
    from naylis_amd.decoder import naylis_config
    from naylis_amd.mom_kernels import hip_rope
    cfg = naylis_config(vocab_size=256, d_model=256, n_layers=1, n_heads=4, intermediate_size=256, seq_len=96)
    attn = hip_rope.NaylisAttention(cfg, 0).to(dev).bfloat16().eval()
    x = torch.randn(2, 96, 256, generator=torch.Generator().manual_seed(0)).bfloat16().to(dev)
    cos, sin = (torch.rand(1, 96, 64, device=dev).bfloat16() for _ in range(2))
    mask = torch.full((96, 96), -math.inf, device=dev).triu(1).bfloat16()[None, None].expand(2, 1, 96, 96)
    assert attn._plain_causal(None, {}) and not attn._plain_causal(mask, {}) and not attn._plain_causal(None, {"x": 1})
    with torch.no_grad():
        got = attn(hidden_states=x, position_embeddings=(cos, sin))[0]
        want = attn(hidden_states=x, position_embeddings=(cos, sin), attention_mask=mask)[0]
    # bf16 P and one rounding of the attention's output each side, then the o projection
    assert float((got.float() - want.float()).norm() / want.float().norm()) < 2.0 ** -7


def test_attention_second_derivative_raises(dev):
    """Gradients taken with create_graph are right (bit for bit the others); a
    second derivative through them raises, also where other paths of the graph
    would go on without it."""
    from naylis_amd.decoder import naylis_config
    from naylis_amd.mom_kernels import hip_rope
    from naylis_amd.mom_kernels.hip_attention import causal_attention
    g = torch.Generator(device=dev).manual_seed(2)
    q, k, v, dout = (torch.randn(1, 70, 2, 64, generator=g, device=dev).bfloat16().requires_grad_() for _ in range(4))
    o = causal_attention(q, k, v, 0.125)
    want = torch.autograd.grad(o, (q, k, v), dout.detach(), retain_graph=True)
    got = torch.autograd.grad(o, (q, k, v), dout, create_graph=True)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    for x in (q, k, v, dout):
        with pytest.raises(RuntimeError, match="not implemented"):
            torch.autograd.grad(sum(t.float().square().sum() for t in got), x, retain_graph=True)
    cfg = naylis_config(vocab_size=256, d_model=128, n_layers=1, n_heads=2, intermediate_size=256, seq_len=96)
    attn = hip_rope.NaylisAttention(cfg, 0).to(dev).bfloat16()
    x = torch.randn(1, 96, 128, generator=g, device=dev).bfloat16().requires_grad_()
    cos, sin = (torch.rand(1, 96, 64, generator=g, device=dev).bfloat16() for _ in range(2))
    dx, = torch.autograd.grad(attn(hidden_states=x, position_embeddings=(cos, sin))[0].float().square().sum(), x,
                              create_graph=True)
    with pytest.raises(RuntimeError, match="not implemented"):
        torch.autograd.grad(dx.float().square().sum(), attn.v_proj.weight)


def test_attention_takes_any_address(dev):
    """Contiguous q, k, v and gradients at addresses that are no multiple of 16
    bytes (views into larger buffers), as torch's attention takes them."""
    from naylis_amd.mom_kernels.hip_attention import causal_attention
    g = torch.Generator(device=dev).manual_seed(4)
    x = [torch.randn(2, 40, 2, 64, generator=g, device=dev).bfloat16() for _ in range(4)]

    def odd(t):
        b = torch.empty(t.numel() + 1, device=dev, dtype=t.dtype)[1:].view(t.shape)
        return b.copy_(t)

    def run(ts):
        q, k, v = (t.requires_grad_() for t in ts[:3])
        o = causal_attention(q, k, v, 0.125)
        return [o, *torch.autograd.grad(o, (q, k, v), ts[3])]

    for a, b in zip(run(x), run([odd(t.detach()) for t in x])):
        assert torch.equal(a, b)


def test_attention_rounds_no_largest_weight(dev):
    """The largest weight, the exponential of the largest score less itself, is
    exactly 1 in bf16. The output's squared error is then that of its own rounding
    plus, for each of the other weights p, that of p's: d^2 p^2 |v|^2 with d the
    mean relative error of rounding, 10 % spared; with the largest weight's the
    error would be a fifth larger on these scores."""
    from naylis_amd.mom_kernels.hip_attention import causal_attention
    g = torch.Generator(device=dev).manual_seed(6)
    q, k, v = (torch.randn(2, 1021, 4, 64, generator=g, device=dev).bfloat16() for _ in range(3))
    q = 3 * q
    o = causal_attention(q, k, v, 0.125).double().transpose(1, 2)
    qd, kd, vd = (t.double().transpose(1, 2) for t in (q, k, v))
    s = qd @ kd.transpose(-1, -2) * 0.125
    s.masked_fill_(torch.ones(1021, 1021, dtype=torch.bool, device=dev).triu(1), -math.inf)
    p = torch.softmax(s, -1)
    ref = p @ vd
    own = (ref.bfloat16().double() - ref).square().sum()
    d2 = (p.bfloat16().double() - p).square().sum() / p.square().sum()
    weights = p.square() @ vd.square().sum(-1, keepdim=True)
    top = p.amax(-1, keepdim=True).square() * vd.square().sum(-1, keepdim=True).gather(2, p.argmax(-1, keepdim=True))
    bound = (own + d2 * (weights - top).sum()).sqrt()
    assert float((own + d2 * weights.sum()).sqrt()) > 1.15 * float(bound)
    assert float((o - ref).norm()) < 1.1 * float(bound)
