"""GPU parity of the LM head's products (klp_lmh_logits, klp_head_dweight,
klp_head_dhidden) against float64 products of the same 16-bit operands.

Each output is a float32 sum of K products, rounded once to the dtype (or kept
in float32): |ours - exact| <= K * 2^-24 * sum_k |a_k b_k| + half an ulp of the
dtype, 2^-p |exact| (2^-25 for subnormal fp16 results)."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
SIG_BITS = {torch.bfloat16: 8, torch.float16: 11, torch.float32: 24}

# Tokens, vocabulary and hidden sizes at and around the 256 x 256 tiles and the
# 64-column stages; several K ranges of d_hidden.
SIZES = [(1, 1, 64), (64, 256, 64), (255, 257, 128), (257, 511, 320), (70, 1000, 192),
         (300, 5003, 576), (2, 70001, 64), (520, 9000, 1024), (190, 70000, 64)]


def _operands(N, V, D, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    h = torch.randn(N, D, generator=g).to(dtype).to(DEV)
    w = (torch.randn(V, D, generator=g) * 0.25).to(dtype).to(DEV)
    ld = -(-V // 8) * 8
    d = torch.zeros(N, ld, dtype=dtype)
    d[:, :V] = torch.randn(N, V, generator=g).to(dtype)
    return h, w, d.to(DEV), ld


def _check(got, exact, mag, K, what):
    p = SIG_BITS[got.dtype]
    bound = K * 2.0 ** -24 * mag + 2.0 ** -p * exact.abs() + 2.0 ** -25
    err = (got.double() - exact).abs()
    assert torch.all(err <= bound), f"{what}: {(err / bound).max().item():.3g}x the bound"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,V,D", SIZES)
def test_products_match_float64(N, V, D, dtype):
    from kernel_opt import _head
    from kernel_opt._library import stream_handle
    h, w, d, ld = _operands(N, V, D, dtype, N + V + D)
    s = stream_handle(0)
    hd, wd, dd = h.double(), w.double(), d[:, :V].double()

    # logits, in rows of any alignment, untouched past their columns
    for pad in (0, 8 - V % 8, 3):
        out = torch.full((N, V + pad), 7.0, dtype=dtype, device=DEV)
        view = out[:, :V] if N > 1 else out.view(-1)[:V].view(1, V)
        _head.logits_into(view, h, w, s)
        torch.cuda.synchronize()
        _check(out[:, :V], hd @ wd.T, hd.abs() @ wd.abs().T, D, f"logits pad {pad}")
        assert torch.all(out[:, V:] == 7.0)

    dw = torch.full((V, D), float("nan"), dtype=dtype, device=DEV)
    _head.d_weight_into(dw, d, ld, h, s)
    _check(dw, dd.T @ hd, dd.abs().T @ hd.abs(), N, "d_weight")

    exact, mag = dd @ wd, dd.abs() @ wd.abs()
    dh = torch.full((N, D), float("nan"), dtype=dtype, device=DEV)
    _head.d_hidden_into(dh, None, False, d, ld, N, w, s)
    _check(dh, exact, mag, V, "d_hidden")
    acc = torch.full((N, D), float("nan"), device=DEV)
    _head.d_hidden_into(None, acc, False, d, ld, N, w, s)
    _check(acc, exact, mag, V, "d_hidden float32")
    _head.d_hidden_into(None, acc, True, d, ld, N, w, s)
    _check(acc, 2 * exact, 2 * mag, V, "d_hidden accumulated")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,V,D", [(200, 33003, 1088), (2500, 9030, 3264)])
def test_products_of_several_tiles_a_workgroup(N, V, D, dtype):
    """More tiles than the 256 workgroups, each of several K stages with
    remainders along every side: the rings run on from one tile to the next.
    d_hidden's tiles come with several K ranges, the last one shorter."""
    from kernel_opt import _head
    from kernel_opt._library import lib, stream_handle
    up = lambda a, b: -(-a // b)  # noqa: E731
    h, w, d, ld = _operands(N, V, D, dtype, N + V + D)
    s = stream_handle(0)
    hd, wd, dd = h.double(), w.double(), d[:, :V].double()
    assert up(D, 256) * up(V, 256) > 256
    dw = torch.full((V, D), float("nan"), dtype=dtype, device=DEV)
    _head.d_weight_into(dw, d, ld, h, s)
    _check(dw, dd.T @ hd, dd.abs().T @ hd.abs(), N, "d_weight")
    splits = lib.klp_head_dhidden_workspace_bytes(N, V, D) // (N * D * 4)
    if N == 2500:
        stages = up(V, 64)
        assert up(D, 256) * up(N, 256) * splits > 256
        assert splits > 1 and stages % up(stages, splits) != 0
    dh = torch.full((N, D), float("nan"), dtype=dtype, device=DEV)
    _head.d_hidden_into(dh, None, False, d, ld, N, w, s)
    _check(dh, dd @ wd, dd.abs() @ wd.abs(), V, "d_hidden")


def test_nan_and_infinity_stay_in_their_rows():
    """A NaN or an infinity among d_logits reaches the output rows it belongs
    to and no other."""
    from kernel_opt import _head
    from kernel_opt._library import stream_handle
    N, V, D = 300, 1100, 192
    h, w, d, ld = _operands(N, V, D, torch.bfloat16, 6)
    s = stream_handle(0)
    for value in (float("nan"), float("inf"), float("-inf")):
        bad = d.clone()
        bad[137, 1001] = value
        dw, dh = torch.empty_like(w), torch.empty_like(h)
        _head.d_weight_into(dw, bad, ld, h, s)
        _head.d_hidden_into(dh, None, False, bad, ld, N, w, s)
        for out, row in ((dw, 1001), (dh, 137)):
            wrong = ~torch.isfinite(out)
            assert wrong[row].all() and wrong.sum() == out.size(1)


def test_strided_operands_and_repeats():
    """Rows with a stride past their columns, garbage (NaN) in the columns
    between; the same bits from one call to the next."""
    from kernel_opt import _head
    from kernel_opt._library import stream_handle
    N, V, D = 130, 1100, 192
    h, w, d, _ = _operands(N, V, D, torch.bfloat16, 5)

    def padded(t, extra):
        big = torch.full((t.size(0), t.size(1) + extra), float("nan"), dtype=t.dtype, device=DEV)
        big[:, :t.size(1)] = t
        return big[:, :t.size(1)]

    hs, ws, ds = padded(h, 8), padded(w, 24), padded(d, 16)
    s = stream_handle(0)
    res = []
    for hh, ww, dd in ((h, w, d), (hs, ws, ds), (hs, ws, ds)):
        lg = torch.empty(N, V, dtype=torch.bfloat16, device=DEV)
        dw, dh = torch.empty_like(w), torch.empty_like(h)
        _head.logits_into(lg, hh, ww, s)
        _head.d_weight_into(dw, dd, dd.stride(0), hh, s)
        _head.d_hidden_into(dh, None, False, dd, dd.stride(0), N, ww, s)
        res.append((lg, dw, dh))
    for other in res[1:]:
        for a, b in zip(res[0], other):
            assert torch.equal(a, b)


def test_rounded_forward_uses_the_written_logits(oracle):
    """The chunked head's one-GEMM forward rounds each logit as klp_lmh_logits
    writes it: the logprob bar on those logits, fp16 and a temperature
    included, and the chunked backward's d_logits from the same."""
    from kernel_opt import _head, fused_linear_logprob_entropy_forward
    from kernel_opt._library import stream_handle
    for dtype, T in ((torch.bfloat16, None), (torch.float16, 0.7)):
        N, V, D = 150, 3001, 256
        h, w, _, _ = _operands(N, V, D, dtype, 9)
        t = torch.arange(N, device=DEV) * 20
        lg = torch.empty(N, V, dtype=dtype, device=DEV)
        _head.logits_into(lg, h, w, stream_handle(0))
        outs = fused_linear_logprob_entropy_forward(h, w, t, T)
        ref = oracle.forward(lg.cpu(), t.cpu().numpy(), temperature=T)
        for o, r in zip(outs, ref):
            assert abs(o.cpu().double().numpy() - r).max() <= 2e-5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,V,row", [(200, 3001, 3000), (200, 3001, 100), (200, 300, 299),
                                     (192, 70001, 70000)])
def test_logits_of_infinity_and_nan(N, V, row, dtype):
    """A weight row that gives some tokens a logit of -inf, some +inf, some NaN,
    in a full tile and in the one at the end: the fold and the gradient as the
    logprob kernels compute them from the same logits.  The fold's sums run in
    another order (2e-5, the bar of both); d_logits round once (2^-7)."""
    import ctypes

    from kernel_opt import (_head, fused_linear_logprob_entropy_forward, fused_logprob_entropy)
    from kernel_opt._library import DTYPE_CODES, check_status, lib, stream_handle
    D = 192
    h, w, _, _ = _operands(N, V, D, dtype, 13)
    w[row, 0] = float("-inf")
    h[:, 0] = torch.tensor([1.0, -1.0, 0.0, 2.0], device=DEV).repeat(N // 4)  # -inf +inf NaN -inf
    t = torch.arange(N, device=DEV) * 7 % V
    t[::5] = row
    x = torch.empty(N, V, dtype=dtype, device=DEV)
    _head.logits_into(x, h, w, stream_handle(0))
    col = x[:, row].float()
    assert torch.isneginf(col[0::4]).all() and torch.isposinf(col[1::4]).all()
    assert torch.isnan(col[2::4]).all()
    g = [torch.linspace(-1, 1, N, device=DEV), torch.linspace(0.5, 1, N, device=DEV),
         torch.linspace(0.1, 0.2, N, device=DEV)]
    for T in (None, 0.7):
        ours = fused_linear_logprob_entropy_forward(h, w, t, T)
        xr = x.clone().requires_grad_(True)
        ref = fused_logprob_entropy(xr, t, T)
        d_ref, = torch.autograd.grad(ref, xr, g)
        for o, r in zip(ours, ref):
            assert torch.equal(o.isnan(), r.isnan()) and torch.equal(o.isinf(), r.isinf())
            live = torch.isfinite(r)
            assert live[0::4].sum() + live[3::4].sum() > 0
            assert torch.all((o - r)[live].abs() <= 4e-5)
        ld = -(-V // 8) * 8
        d = torch.empty(N, ld, dtype=dtype, device=DEV)
        P = lambda a: ctypes.c_void_p(a.data_ptr())  # noqa: E731
        check_status(lib.klp_lmh_bwd_logits_as(
            DTYPE_CODES[dtype], 1, P(h), D, P(w), D, N, V, D, P(t), 0, T or 1.0, P(ref[2]),
            P(ref[1]), P(g[0]), P(g[1]), P(g[2]), P(d), ld, stream_handle(0)))
        d = d[:, :V]
        assert torch.equal(d.isnan(), d_ref.isnan()) and torch.equal(d.isinf(), d_ref.isinf())
        live = torch.isfinite(d_ref)
        a, b = d[live].float(), d_ref[live].float()
        assert live.any() and torch.all((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-6)


def test_library_rule_boundaries():
    """The chunked head's backward with d_hidden and d_weight through the
    kernels, through the library, and with one of each: the same gradients up
    to the rounding of the operands' dtype."""
    from kernel_opt import _head, fused_linear_logprob_entropy
    N, V, D = 96, 4099, 128
    h, w, _, _ = _operands(N, V, D, torch.bfloat16, 11)
    t = torch.arange(N, device=DEV) * 40
    g = torch.linspace(-1, 1, N, device=DEV)
    res = []
    saved = _head.d_hidden_pays, _head.d_weight_pays
    from kernel_opt import lmhead
    try:
        for own_h, own_w in ((True, True), (False, False), (True, False), (False, True)):
            lmhead.d_hidden_pays = lambda *a: own_h
            lmhead.d_weight_pays = lambda *a: own_w
            ha, wa = h.clone().requires_grad_(True), w.clone().requires_grad_(True)
            lp, ent, _ = fused_linear_logprob_entropy(ha, wa, t, chunk_vocab=1500)
            res.append(torch.autograd.grad((lp, ent), (ha, wa), (g, 0.1 * g)))
    finally:
        lmhead.d_hidden_pays, lmhead.d_weight_pays = saved
    for other in res[1:]:
        for a, b in zip(res[0], other):
            # one rounding to bf16 each, of equal float32 sums up to their order
            assert ((a.float() - b.float()).abs() <= 2.0 ** -7 * a.float().abs() + 1e-6).all()
