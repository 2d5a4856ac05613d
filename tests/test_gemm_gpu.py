"""GPU checks of the split-K MFMA GEMM behind the q/o projection weight
gradient (C ABI naylis_mom_linear_wgrad; model.py:239,251 take it from
autograd as dy^T x over all tokens) against an fp64 product of the same bf16
inputs, plus the autograd binding against torch's own linear.

Tolerance: |got - ref| <= 2e-2 |ref| + 2e-3 max(1, max|ref|) (a sum over up to
16384 tokens has magnitudes >> 1; the atol scales with it as for the other
parameter gradients); results must be bitwise reproducible.
"""
import copy

import pytest
import torch

from tests._tol import assert_close

pytestmark = pytest.mark.gpu


def wgrad(x, dy, out_dtype):
    from naylis_amd import _lib
    lib = _lib.load()
    N, D_in = x.shape
    D_out = dy.shape[1]
    ws = torch.empty(lib.naylis_mom_linear_wgrad_workspace_bytes(N, D_in, D_out), device=x.device, dtype=torch.uint8)
    dw = torch.full((D_out, D_in), float("nan"), device=x.device, dtype=out_dtype)
    rc = lib.naylis_mom_linear_wgrad(x.data_ptr(), dy.data_ptr(), dw.data_ptr(), 0 if out_dtype == torch.float32 else 1,
                                     ws.data_ptr(), ws.numel(), N, D_in, D_out,
                                     torch.cuda.current_stream().cuda_stream)
    _lib.check(rc)
    return dw


@pytest.mark.parametrize("N,D_in,D_out,out_dtype", [
    (16384, 1024, 1024, torch.bfloat16),   # config 2: B*T tokens, d x d
    (16384, 1024, 1024, torch.float32),
    (16384, 1536, 1536, torch.bfloat16),   # config 4 width
    (1000, 64, 192, torch.float32),        # ragged token count, rectangular
    (8, 24, 40, torch.float32),            # below one tile in every dimension
])
def test_linear_wgrad_matches_fp64(N, D_in, D_out, out_dtype, dev):
    g = torch.Generator().manual_seed(N + D_in)
    x = torch.randn(N, D_in, generator=g).bfloat16()
    dy = torch.randn(N, D_out, generator=g).bfloat16()
    got = wgrad(x.to(dev), dy.to(dev), out_dtype)
    torch.cuda.synchronize()
    ref = dy.double().T @ x.double()
    assert_close(got, ref, "dW", atol=2e-3 * max(1.0, float(ref.abs().max())))


def test_linear_wgrad_deterministic_and_empty(dev):
    g = torch.Generator().manual_seed(3)
    x = torch.randn(16384, 1024, generator=g).bfloat16().to(dev)
    dy = torch.randn(16384, 1024, generator=g).bfloat16().to(dev)
    a = wgrad(x, dy, torch.float32)
    b = wgrad(x, dy, torch.float32)
    assert torch.equal(a, b)
    z = wgrad(x[:0], dy[:0], torch.float32)
    torch.cuda.synchronize()
    assert torch.equal(z.cpu(), torch.zeros(1024, 1024))


def test_mom_linear_autograd_matches_torch(dev):
    from naylis_amd import mom_kernels
    g = torch.Generator().manual_seed(4)
    x = torch.randn(4, 512, 256, generator=g).bfloat16().to(dev).requires_grad_(True)
    w = (torch.randn(384, 256, generator=g) * 0.05).bfloat16().to(dev).requires_grad_(True)
    dy = torch.randn(4, 512, 384, generator=g).bfloat16().to(dev)
    y = mom_kernels.mom_linear(x, w)
    y.backward(dy)
    xr = x.detach().double().requires_grad_(True)
    wr = w.detach().double().requires_grad_(True)
    yr = torch.nn.functional.linear(xr, wr)
    yr.backward(dy.double())
    assert_close(y, yr, "y")
    assert_close(x.grad, xr.grad, "dx")
    assert_close(w.grad, wr.grad, "dW", atol=2e-3 * max(1.0, float(wr.grad.abs().max())))


def test_naylis_linear_module_swap(dev):
    """use_library_wgrad turns the bias-free nn.Linear of a block into
    NaylisLinear in place: same parameters and keys, the same forward and
    input gradient as nn.Linear, the weight gradient from the library (to the
    bf16 GEMM bound); a biased Linear is left alone."""
    from naylis_amd.mom_kernels.hip_linear import NaylisLinear, use_library_wgrad
    torch.manual_seed(7)
    block = torch.nn.Sequential(torch.nn.Linear(256, 704, bias=False), torch.nn.Linear(704, 256, bias=True))
    block = block.to(dev, torch.bfloat16)
    ref = copy.deepcopy(block)
    keys = list(block.state_dict())
    use_library_wgrad(block)
    assert type(block[0]) is NaylisLinear and type(block[1]) is torch.nn.Linear
    assert list(block.state_dict()) == keys
    x = torch.randn(2, 512, 256, device=dev, dtype=torch.bfloat16)
    dy = torch.randn(2, 512, 256, device=dev, dtype=torch.bfloat16)
    xa, xb = x.clone().requires_grad_(True), x.clone().requires_grad_(True)
    ya = block(xa)
    ya.backward(dy)
    hb = ref[0](xb)
    hb.retain_grad()
    yb = ref[1](hb)
    yb.backward(dy)
    assert torch.equal(ya, yb)
    assert_close(xa.grad, xb.grad, "dx")
    # the first layer's exact weight gradient from the bf16 gradient reaching it
    gw = torch.mm(hb.grad.reshape(-1, 704).float().t(), x.reshape(-1, 256).float())
    # bf16 output rounding (half an ulp, at most 2^-8 relative) plus the accumulation
    tol = 2.0 ** -8 * gw.abs() + 2e-3 * max(1.0, float(gw.abs().max()))
    assert bool(((block[0].weight.grad.float() - gw).abs() <= tol).all())
    assert bool(((ref[0].weight.grad.float() - gw).abs() <= tol).all())
    assert_close(block[1].weight.grad, ref[1].weight.grad, "dW (nn.Linear)")


def test_shared_input_linear_matches_separate_layers(dev):
    """shared_input_linear (q/k/v, gate/up of the decoder): the same outputs as
    applying the layers one by one; the input gradient is the sum of the
    products accumulated in one GEMM epilogue (close to autograd's sum of
    rounded products), weight gradients to the bf16 GEMM bound."""
    from naylis_amd.mom_kernels.hip_linear import shared_input_linear
    torch.manual_seed(11)
    layers = [torch.nn.Linear(256, n, bias=False).to(dev, torch.bfloat16) for n in (256, 512, 256)]
    x = torch.randn(2, 512, 256, device=dev, dtype=torch.bfloat16)
    dys = [torch.randn(2, 512, m.out_features, device=dev, dtype=torch.bfloat16) for m in layers]
    xa = x.clone().requires_grad_(True)
    outs = shared_input_linear(xa, layers)
    torch.autograd.backward(outs, dys)
    wgrads = [m.weight.grad.clone() for m in layers]
    for m in layers:
        m.weight.grad = None
    for o, m in zip(outs, layers):
        assert torch.equal(o, m(x))
    x32 = x.reshape(-1, 256).float()
    parts = [torch.mm(d.reshape(-1, m.out_features).float(), m.weight.detach().float()) for d, m in zip(dys, layers)]
    dx = sum(parts)
    # three bf16 roundings of partial sums (here, and in autograd's sum of rounded products), each at most
    # 2^-9 of the sum of the products' magnitudes, plus the GEMMs' accumulation
    tol = 2.0 ** -7 * sum(q.abs() for q in parts) + 1e-3
    assert bool(((xa.grad.reshape(-1, 256).float() - dx).abs() <= tol).all())
    # and no further from the fp32 sum than autograd's own sum over the separate layers
    xb = x.clone().requires_grad_(True)
    torch.autograd.backward([m(xb) for m in layers], dys)
    err_lib = float((xa.grad.reshape(-1, 256).float() - dx).abs().max())
    err_torch = float((xb.grad.reshape(-1, 256).float() - dx).abs().max())
    assert err_lib <= 1.5 * err_torch + 1e-3, (err_lib, err_torch)
    for d, m, g in zip(dys, layers, wgrads):
        gw = torch.mm(d.reshape(-1, m.out_features).float().t(), x32)
        tol = 2.0 ** -8 * gw.abs() + 2e-3 * max(1.0, float(gw.abs().max()))
        assert bool(((g.float() - gw).abs() <= tol).all())
    # no grad: the plain layers
    with torch.no_grad():
        outs = shared_input_linear(x, layers)
    assert all(o.grad_fn is None for o in outs)


def _sum_bound(a, b, ref):
    """A bf16 result of an fp32 sum of n products: one bf16 rounding (2^-8
    relative) and sqrt(n) fp32 roundings of the terms' magnitudes, eight fold."""
    n = a.shape[1]
    return 2.0 ** -8 * ref.abs() + 8 * n ** 0.5 * 2.0 ** -24 * (a.abs() @ b.abs())


@pytest.mark.parametrize("N,D_in,D_out", [
    (16384, 1000, 1032),   # K ranges, last tiles of 104 columns and 8 rows
    (9952, 1024, 1024),    # 311 steps a tile, listed as 312: empty last steps
    (12288, 128, 3064),    # one column of tiles
    (16384, 2816, 264),    # one band of two columns left over, 8 rows past a tile
    (2048, 5632, 2048),    # whole K per tile, 256 x 256 tiles
    (1024, 4104, 2056),    # the same with edges in both directions
])
def test_linear_wgrad_pipelined_shapes(N, D_in, D_out, dev):
    g = torch.Generator(device=dev).manual_seed(D_in)
    x = torch.randn(N, D_in, generator=g, device=dev).bfloat16()
    dy = torch.randn(N, D_out, generator=g, device=dev).bfloat16()
    got = wgrad(x, dy, torch.bfloat16).double()
    a, b = dy.double().t(), x.double()
    ref = a @ b
    assert bool(((got - ref).abs() <= _sum_bound(a, b, ref)).all())
    assert torch.equal(got, wgrad(x, dy, torch.bfloat16).double())


@pytest.mark.parametrize("L,D", [(4000, 1568), (2048, 2048), (3000, 2080)])
def test_bank_kv_pipelined_shapes(L, D, dev):
    """The bank projection's three layouts on the pipelined tiles (the two K
    segments of d_slots included), with edge tiles."""
    from naylis_amd.mom_kernels.hip_bank import mom_bank_kv
    g = torch.Generator(device=dev).manual_seed(L)
    s, dk, dv = (torch.randn(L, D, generator=g, device=dev).bfloat16() for _ in range(3))
    wk, wv = (torch.randn(D, D, generator=g, device=dev).bfloat16() for _ in range(2))
    s, wk, wv = (t.requires_grad_() for t in (s, wk, wv))
    k, v = mom_bank_kv(s, wk, wv)
    torch.autograd.backward([k, v], [dk, dv])
    s, wk, wv, k, v, dk, dv, ds, dwk, dwv = (t.detach().double() for t in (s, wk, wv, k, v, dk, dv, s.grad, wk.grad,
                                                                           wv.grad))
    for got, a, b in ((k, s, wk.t()), (v, s, wv.t()), (ds, torch.cat([dk, dv], 1), torch.cat([wk, wv], 0)),
                      (dwk, dk.t(), s), (dwv, dv.t(), s)):
        ref = a @ b
        assert bool(((got - ref).abs() <= _sum_bound(a, b, ref)).all())


def test_gated_wgrad_pipelined(dev):
    """The gate epilogue on K ranges: dW = s dW', ds = sum dW' W."""
    from naylis_amd.mom_kernels.hip_rezero import mom_gated_linear
    g = torch.Generator(device=dev).manual_seed(0)
    N, D = 16384, 1024
    x, dy = (torch.randn(N, D, generator=g, device=dev).bfloat16() for _ in range(2))
    w = (torch.randn(D, D, generator=g, device=dev) / 32).bfloat16().requires_grad_()
    s = torch.full((1,), 0.75, device=dev, requires_grad=True)
    mom_gated_linear(x, w, s).backward(dy.float())
    a, b = dy.double().t(), x.double()
    ref = a @ b
    assert bool(((w.grad.double() - 0.75 * ref).abs() <= _sum_bound(a, b, 0.75 * ref)).all())
    # a million products of dW' (each within 8 sqrt(n) roundings, independent) and W
    ds = (ref * w.detach().double()).sum()
    var = ((8 * N ** 0.5 * 2.0 ** -24 * (a.abs() @ b.abs())) * w.detach().double()).square().sum().sqrt()
    assert abs(float(s.grad) - float(ds)) <= float(var) + 2.0 ** -20 * float((ref * w.detach().double()).abs().sum())


@pytest.mark.parametrize("N", [1, 63, 64, 131, 1021, 2048, 2050])
@pytest.mark.parametrize("D_in,D_out,n", [(64, 128, 3), (1024, 1024, 3), (1024, 2816, 2), (2816, 1024, 1),
                                          (256, 640, 2)])
def test_linear_fwd_and_dgrad_match_fp64(N, D_in, D_out, n, dev):
    """naylis_mom_linear_fwd (one to three weights, bf16 and fp32 results) and
    naylis_mom_linear_dgrad at row counts around the tiles, odd ones among them."""
    import ctypes

    from naylis_amd import _lib
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev).manual_seed(N + D_in)
    x = torch.randn(N, D_in, generator=g, device=dev).bfloat16()
    dy = torch.randn(N, D_out, generator=g, device=dev).bfloat16()
    ws = [torch.randn(D_out, D_in, generator=g, device=dev).bfloat16() for _ in range(n)]
    ptrs = lambda ts: (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])  # noqa: E731
    for code, dtype in ((0, torch.float32), (1, torch.bfloat16)):
        ys = [torch.full((N + 1, D_out), 7.0, device=dev, dtype=dtype) for _ in range(n)]
        _lib.check(lib.naylis_mom_linear_fwd(x.data_ptr(), ptrs(ws), ptrs(ys), n, code, N, D_in, D_out, st))
        for y, w in zip(ys, ws):
            a, b = x.double(), w.double().t()
            ref = a @ b
            bound = _sum_bound(a, b, ref)
            assert bool(((y[:N].double() - ref).abs() <= bound).all())
            assert bool((y[N] == 7).all())      # nothing past the last row
    dx = torch.full((N + 1, D_in), 7.0, device=dev, dtype=torch.bfloat16)
    _lib.check(lib.naylis_mom_linear_dgrad(dy.data_ptr(), ws[0].data_ptr(), dx.data_ptr(), N, D_in, D_out, st))
    a, b = dy.double(), ws[0].double()
    ref = a @ b
    assert bool(((dx[:N].double() - ref).abs() <= _sum_bound(a, b, ref)).all()) and bool((dx[N] == 7).all())


def test_linear_routes(dev):
    """Evaluation and training take the same product (bit for bit) at a token
    count that is a multiple of 8; transforms, tracing and module hooks keep
    torch's."""
    from naylis_amd.mom_kernels.hip_linear import NaylisLinear, shared_input_linear
    g = torch.Generator(device=dev).manual_seed(1)
    mods = [NaylisLinear(256, 384, bias=False).to(dev, torch.bfloat16) for _ in range(3)]
    x = torch.randn(3, 80, 256, generator=g, device=dev).bfloat16()
    train = shared_input_linear(x, mods)
    want = [torch.nn.functional.linear(x.double(), m.weight.double()) for m in mods]
    with torch.no_grad():
        ev = shared_input_linear(x, mods)
        assert all(torch.equal(a, b) for a, b in zip(train, ev))
        for y, r, m in zip(ev, want, mods):
            a, b = x.double().view(-1, 256), m.weight.double().t()
            assert bool(((y.double() - r).abs() <= _sum_bound(a, b, r.view(-1, 384)).view_as(r)).all())
        mapped = torch.func.vmap(mods[0])(x)
        assert mapped.shape == ev[0].shape
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
            assert torch.autograd.forward_ad.unpack_dual(mods[0](dual)).tangent is not None
        seen = []
        h = mods[1].register_forward_hook(lambda m, i, o: seen.append(1))
        shared_input_linear(x, mods)
        h.remove()
        assert seen == [1]
        traced = torch.jit.trace(mods[0], (x,), check_trace=False)
        assert not torch.equal(traced(x), traced(2 * x))


@pytest.mark.parametrize("N,D_in,D_out,fwd,dgrad", [
    (1400, 1024, 2816, True, True),     # 242 tiles of 128 x 128: one round
    (1533, 1024, 2816, False, True),    # 264 and 132 of 256 x 128: between (dx: 1533 x 1024, 96 tiles)
    (1533, 2816, 1024, True, False),    # the same for dx
    (1661, 1024, 2816, True, True),     # 286 and 154
])
def test_linear_leaves_between_tiles_to_torch(N, D_in, D_out, fwd, dgrad, dev):
    """Products that neither the one-round tiles nor the large ones take stay on
    torch's GEMM (the kernels that ran, by their timer's names)."""
    from naylis_amd import _lib, _torch_ext
    x, dy = (torch.ones(N, d, device=dev, dtype=torch.bfloat16) for d in (D_in, D_out))
    w = torch.ones(D_out, D_in, device=dev, dtype=torch.bfloat16)
    ext, st = _torch_ext.load(), _lib.stream_of(dev)
    with _lib.KernelTimer():
        ext.linear(x, [w], False, st)
        ext.linear_dgrad(dy, w, st)
    names = _lib.KernelTimer.results()
    assert ("linear_fwd" in names, "linear_dgrad" in names) == (fwd, dgrad)


@pytest.mark.parametrize("grad", [False, True])
def test_linear_of_no_features(grad, dev):
    """Layers of no input features give zeros, as torch's do."""
    from naylis_amd.mom_kernels.hip_linear import mom_linear, shared_input_linear
    mods = [torch.nn.Linear(8, 16, bias=False).to(dev, torch.bfloat16) for _ in range(2)]
    for m in mods:
        m.weight = torch.nn.Parameter(m.weight.detach()[:, :0])
    x = torch.zeros(8, 0, device=dev, dtype=torch.bfloat16)
    with torch.set_grad_enabled(grad):
        ys = [mom_linear(x, mods[0].weight), *shared_input_linear(x, mods)]
    assert all(torch.equal(y, torch.zeros(8, 16, device=dev, dtype=torch.bfloat16)) for y in ys)


def test_linear_keeps_global_hooks_and_replaced_forwards(dev):
    from naylis_amd.mom_kernels.hip_linear import NaylisLinear, shared_input_linear
    mods = [NaylisLinear(256, 384, bias=False).to(dev, torch.bfloat16) for _ in range(2)]
    x = torch.randn(16, 256, device=dev).bfloat16()
    with torch.no_grad():
        seen = []
        h = torch.nn.modules.module.register_module_forward_hook(lambda m, i, o: seen.append(m))
        shared_input_linear(x, mods)
        h.remove()
        assert seen == mods
        mods[1].forward = lambda x: torch.zeros(1)
        assert shared_input_linear(x, mods)[1].numel() == 1


def test_linear_second_derivative(dev):
    """A gradient taken with create_graph: the input gradient g = dy W stays a
    product that autograd knows, d(sum(g^2) / 2)/d dy = g W^T."""
    from naylis_amd import mom_kernels
    g = torch.Generator(device=dev).manual_seed(3)
    x = torch.randn(128, 256, generator=g, device=dev).bfloat16().requires_grad_(True)
    w = (torch.randn(384, 256, generator=g, device=dev) * 0.05).bfloat16().requires_grad_(True)
    dy = torch.randn(128, 384, generator=g, device=dev).bfloat16().requires_grad_(True)
    dx, = torch.autograd.grad(mom_kernels.mom_linear(x, w), x, dy, create_graph=True)
    got, = torch.autograd.grad(dx, dy, dx.detach())
    a, b = dx.detach().double(), w.detach().double().t()
    ref = a @ b
    assert bool(((got.double() - ref).abs() <= _sum_bound(a, b, ref)).all())


@pytest.mark.parametrize("grad", [False, True])
def test_traced_modules_follow_their_input(grad, dev):
    """A traced norm and projection run their kernels on the inputs of each call
    (bit for bit the eager results, gradients among them)."""
    from naylis_amd.mom_kernels.hip_linear import NaylisLinear
    from naylis_amd.mom_kernels.hip_norm import NaylisRMSNorm
    block = torch.nn.Sequential(NaylisRMSNorm(512), NaylisLinear(512, 512, bias=False)).to(dev, torch.bfloat16)
    g = torch.Generator(device=dev).manual_seed(5)
    a, b = (torch.randn(64, 512, generator=g, device=dev).bfloat16().requires_grad_(grad) for _ in range(2))
    with torch.set_grad_enabled(grad):
        traced = torch.jit.trace(block, (a,), check_trace=False)
        y, want = traced(b), block(b)
        assert torch.equal(y, want)
        if grad:
            ins = (b, *block.parameters())
            for p, q in zip(torch.autograd.grad(y, ins, y.detach()), torch.autograd.grad(want, ins, y.detach())):
                assert torch.equal(p, q)


@pytest.mark.parametrize("rows,cols", [(500, 1000), (500, 2824), (1000, 2824),  # 64 x 64, 64 x 128, 128 x 128 tiles
                                       (4100, 2824)])                           # 192 x 256, 256 x 128
@pytest.mark.parametrize("K", [64, 576])                                           # one step; more than any ring holds
def test_small_tiles(rows, cols, K, dev):
    """One-round products on the small pipelined tiles, ragged in both directions,
    in the three operand layouts: weight gradient, forward and input gradient."""
    import ctypes

    from naylis_amd import _lib
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev).manual_seed(rows + cols + K)
    r8 = rows // 8 * 8
    a = torch.randn(rows, K, generator=g, device=dev).bfloat16()
    w = torch.randn(cols, K, generator=g, device=dev).bfloat16()
    ref = a.double() @ w.double().t()
    bound = _sum_bound(a.double(), w.double().t(), ref)
    got = wgrad(w.t().contiguous(), a[:r8].t().contiguous(), torch.bfloat16).double()
    assert bool(((got - ref[:r8]).abs() <= bound[:r8]).all())
    y, dx = (torch.full((rows + 1, cols), 7.0, device=dev, dtype=torch.bfloat16) for _ in range(2))
    _lib.check(lib.naylis_mom_linear_fwd(a.data_ptr(), (ctypes.c_void_p * 1)(w.data_ptr()),
                                         (ctypes.c_void_p * 1)(y.data_ptr()), 1, 1, rows, K, cols, st))
    wt = w.t().contiguous()
    _lib.check(lib.naylis_mom_linear_dgrad(a.data_ptr(), wt.data_ptr(), dx.data_ptr(), rows, cols, K, st))
    for out in (y, dx):
        assert bool(((out[:rows].double() - ref).abs() <= bound).all()) and bool((out[rows] == 7).all())


@pytest.mark.parametrize("N", [1, 61, 3885, 16381])
@pytest.mark.parametrize("D_in,D_out", [(1024, 1024), (264, 520), (2824, 1000)])
def test_linear_wgrad_rows(N, D_in, D_out, dev):
    """Row counts that are no multiple of 8: one tile per workgroup, K splits and K ranges."""
    from naylis_amd import _lib
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev).manual_seed(N + D_in)
    # the next rows hold infinities: none may be read into a sum
    x, dy = (torch.cat([torch.randn(N, d, generator=g, device=dev), torch.full((64, d), float("inf"), device=dev)])
             .bfloat16() for d in (D_in, D_out))
    nb = lib.naylis_mom_linear_wgrad_rows_workspace_bytes(N, D_in, D_out)
    ws = torch.empty(nb, dtype=torch.uint8, device=dev)
    a, b = dy[:N].double().t(), x[:N].double()
    ref = a @ b
    for code, dtype in ((0, torch.float32), (1, torch.bfloat16)):
        dw = torch.empty(D_out, D_in, device=dev, dtype=dtype)
        _lib.check(lib.naylis_mom_linear_wgrad_rows(x.data_ptr(), dy.data_ptr(), dw.data_ptr(), code, ws.data_ptr(), nb,
                                                    N, D_in, D_out, st))
        assert bool(((dw.double() - ref).abs() <= _sum_bound(a, b, ref)).all())
