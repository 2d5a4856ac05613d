"""Fused next-token cross-entropy (naylis_mom_xent_*) against the reference's
F.cross_entropy(logits.float(), labels, reduction="sum") (model.py:536-545)
on the same GPU inputs: loss and the bf16 gradient of the logits."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,V", [(4095, 32768), (7, 2048), (300, 6144)])
def test_xent_matches_cross_entropy(N, V, dev):
    from naylis_amd.mom_kernels.hip_xent import cross_entropy_rows
    g = torch.Generator().manual_seed(N)
    logits = (torch.randn(N, V, generator=g) * 4).bfloat16().to(dev)
    labels = torch.randint(0, V, (N,), generator=g)
    labels[::5] = -100                                  # ignored rows
    labels = labels.to(dev)
    n_valid = (labels != -100).sum()
    lr = logits.clone().requires_grad_(True)
    want = F.cross_entropy(lr.float(), labels, reduction="sum") / n_valid
    want.backward()
    lg = logits.clone().requires_grad_(True)
    rows = cross_entropy_rows(lg, labels)
    got = rows.sum() / n_valid
    got.backward()
    torch.cuda.synchronize()
    assert abs(float(got) - float(want)) <= 1e-5 * abs(float(want))
    assert bool((rows[labels == -100] == 0).all())
    # per-row: the fp32 log-sum-exp to a few ulps, then one bf16 rounding of the gradient
    err = (lg.grad.float() - lr.grad.float()).abs()
    bound = lr.grad.float().abs() * 2.0 ** -7 + 1e-9
    assert bool((err <= bound).all()), float((err - bound).max())
    assert bool((lg.grad[labels == -100] == 0).all())


def test_xent_out_of_range_label_is_nan(dev):
    """A label outside [0, V) that is not ignore_index (F.cross_entropy
    raises on it) makes that row's loss and gradient NaN; the other rows are
    unaffected, so the summed loss is NaN rather than silently smaller."""
    from naylis_amd.mom_kernels.hip_xent import cross_entropy_rows
    g = torch.Generator().manual_seed(3)
    N, V = 6, 2048
    logits = (torch.randn(N, V, generator=g) * 4).bfloat16().to(dev)
    labels = torch.randint(0, V, (N,), generator=g)
    labels[1], labels[4] = V, -100                       # one out of range, one ignored
    labels = labels.to(dev)
    lg = logits.clone().requires_grad_(True)
    rows = cross_entropy_rows(lg, labels)
    rows.sum().backward()
    torch.cuda.synchronize()
    assert torch.isnan(rows[1]) and torch.isnan(rows.sum())
    assert float(rows[4]) == 0.0
    ok = torch.tensor([0, 2, 3, 5], device=dev)
    want = F.cross_entropy(logits[ok].float(), labels[ok], reduction="none")
    assert torch.allclose(rows[ok], want, rtol=1e-5, atol=1e-5)
    assert bool(torch.isnan(lg.grad[1]).all()) and bool((lg.grad[4] == 0).all())
    assert bool(torch.isfinite(lg.grad[ok]).all())


def test_xent_rejects_unsupported(dev):
    from naylis_amd.mom_kernels.hip_xent import cross_entropy_rows
    with pytest.raises(RuntimeError, match="multiple of"):
        cross_entropy_rows(torch.randn(4, 1000, device=dev).bfloat16(), torch.zeros(4, dtype=torch.long, device=dev))


@pytest.mark.parametrize("chunks", [1, 2, 3, 4, 5, 8, 9, 17])
def test_xent_forward_masked_rows(chunks, dev):
    """Rows around the forward's register tiles (4 or 8 chunks of 2048), with
    -inf and lowest-value masks over whole threads, chunks and rows, against
    fp64.  The sum's terms carry a relative error of at most (|x - m| + 2) 2^-23
    and |x - m| e^(x - m) is at most 1/e, so the log-sum-exp is within 2^-21 of
    a logarithm plus its own rounding, 2^-23 |loss| with the label's."""
    from naylis_amd.mom_kernels.hip_xent import cross_entropy_rows
    V = 2048 * chunks
    x = (torch.randn(6, V, generator=torch.Generator().manual_seed(chunks)) * 5).bfloat16()
    x[1, 1:] = -float("inf")                   # one finite value
    x[2, : V - 100] = torch.finfo(torch.bfloat16).min
    x[3] = torch.finfo(torch.bfloat16).min     # a row of the lowest value: log V
    x[4, : V // 2] = -float("inf")
    x[5] = 200 * x[5]                          # the largest value decides
    labels = torch.tensor([3, 0, V - 1, 7, V - 1, int(x[5].argmax())])
    want = -torch.log_softmax(x.double(), -1).gather(1, labels[:, None])[:, 0]
    got = cross_entropy_rows(x.to(dev), labels.to(dev)).double().cpu()
    scale = x.double().gather(1, labels[:, None])[:, 0].abs() + want.abs()
    scale[3] = float(torch.finfo(torch.bfloat16).max)  # lse and the label's logit are this large and cancel
    assert bool(((got - want).abs() <= 2.0 ** -21 + 2.0 ** -22 * scale).all()), (got, want)
    x[0] = -float("inf")                       # nothing to choose from: NaN, as log_softmax
    assert bool(cross_entropy_rows(x.to(dev), labels.to(dev))[0].isnan())


@pytest.mark.parametrize("V", [2048, 24576])
def test_xent_gradients_of_unlikely_classes(V, dev):
    """Logits of deviation 40: gradients down to bf16's subnormal range, each within
    a bf16 rounding (2^-8, or half of the subnormal spacing 2^-133) of fp64 and p's
    own error.  That is the row's log-sum-exp, under 2^8, rounded to fp32, 2^-17
    at most, and few ulp of the exponential; a value lies so near a rounding
    boundary that it may go the other way with probability 2 * 2^-17 / 2^-8."""
    from naylis_amd.mom_kernels.hip_xent import cross_entropy_rows
    g = torch.Generator(device=dev).manual_seed(V)
    z = (torch.randn(256, V, generator=g, device=dev) * 40).bfloat16().requires_grad_(True)
    y = torch.randint(0, V, (256,), generator=g, device=dev)
    cross_entropy_rows(z, y).sum().backward()
    logp = torch.log_softmax(z.detach().double(), -1)
    assert float((z.detach().double() - logp).max()) < 2 ** 8
    p = logp.exp()  # (torch's softmax drops values under e^-87 here)
    d = p.scatter_add(1, y[:, None], -torch.ones_like(y[:, None], dtype=p.dtype))
    err = (z.grad.double() - d).abs()
    assert bool((err <= 2.0 ** -8 * d.abs() + 2.0 ** -16 * p + 2.0 ** -134).all())
    assert float((z.grad != d.bfloat16()).double().mean()) < 2.0 ** -8
    assert bool(((z.grad != 0) & (z.grad.abs() < 2.0 ** -126)).any())
