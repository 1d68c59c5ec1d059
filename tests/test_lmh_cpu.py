"""CPU pins of the float64 LM-head oracle (oracle/lmh_oracle.py)."""
from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from oracle import lmh_oracle


def bf16_bits(x: np.ndarray) -> np.ndarray:
    return torch.from_numpy(np.asarray(x, np.float32)).to(torch.bfloat16).view(torch.int16) \
        .numpy().view(np.uint16)


def test_matches_c_oracle_on_exact_integer_logits(oracle):
    """Small-integer hidden / weight: every logit is an integer below 2^24,
    exact in fp32, so the C oracle of the logprob forward sees the same
    logits and must agree to float64 rounding."""
    g = np.random.default_rng(1)
    N, V, D = 9, 777, 64
    h = bf16_bits(g.integers(-3, 4, (N, D)))
    w = bf16_bits(g.integers(-2, 3, (V, D)))
    t = g.integers(-2, V + 2, N)
    lp, ent, lse = lmh_oracle.forward(h, w, t)
    x = lmh_oracle.logits(h, w).astype(np.float32)
    assert np.array_equal(x.astype(np.float64), lmh_oracle.logits(h, w))
    r_lp, r_ent, r_lse = oracle.forward(x, t, dtype="fp32")
    np.testing.assert_allclose(lp, r_lp, rtol=0, atol=1e-12)
    np.testing.assert_allclose(ent, r_ent, rtol=0, atol=1e-12)
    np.testing.assert_allclose(lse, r_lse, rtol=0, atol=1e-12)


def test_matches_python_loop():
    g = np.random.default_rng(2)
    N, V, D = 3, 7, 64
    h = bf16_bits(g.normal(0, 1, (N, D)))
    w = bf16_bits(g.normal(0, 0.3, (V, D)))
    t = np.array([0, 6, 3])
    lp, ent, lse = lmh_oracle.forward(h, w, t, temperature=0.7)
    hf, wf = lmh_oracle.bf16_to_f64(h), lmh_oracle.bf16_to_f64(w)
    s = float(np.float32(1 / 0.7))
    for n in range(N):
        xs = [math.fsum(hf[n, k] * wf[v, k] for k in range(D)) * s for v in range(V)]
        m = max(xs)
        z = math.fsum(math.exp(x - m) for x in xs)
        l = m + math.log(z)
        e = l - math.fsum(math.exp(x - l) * x for x in xs)
        assert abs(lse[n] - l) < 1e-12 and abs(ent[n] - e) < 1e-12
        assert abs(lp[n] - (xs[t[n]] - l)) < 1e-12


def test_uniform_rows_closed_form():
    g = np.random.default_rng(3)
    N, V, D = 4, 1000, 128
    h = bf16_bits(g.normal(0, 1, (N, D)))
    w = np.tile(bf16_bits(g.normal(0, 0.1, (1, D))), (V, 1))
    lp, ent, lse = lmh_oracle.forward(h, w, np.zeros(N, np.int64))
    np.testing.assert_allclose(ent, math.log(V), rtol=0, atol=1e-12)
    np.testing.assert_allclose(lp, -math.log(V), rtol=0, atol=1e-12)


def test_out_of_range_targets_give_minus_lse():
    g = np.random.default_rng(4)
    h = bf16_bits(g.normal(0, 1, (3, 64)))
    w = bf16_bits(g.normal(0, 0.2, (50, 64)))
    lp, _, lse = lmh_oracle.forward(h, w, np.array([-100, 50, 1000]))
    np.testing.assert_array_equal(lp, -lse)


def test_backward_matches_float64_autograd():
    g = np.random.default_rng(5)
    N, V, D = 6, 40, 64
    h = bf16_bits(g.normal(0, 1, (N, D)))
    w = bf16_bits(g.normal(0, 0.3, (V, D)))
    t = np.array([0, 39, 5, -100, 17, 40])
    gl, ge, gs = (g.normal(0, 1, N) for _ in range(3))
    T = 0.8
    dh, dw, _ = lmh_oracle.backward(h, w, t, gl, ge, gs, temperature=T)
    H = torch.tensor(lmh_oracle.bf16_to_f64(h), requires_grad=True)
    W = torch.tensor(lmh_oracle.bf16_to_f64(w), requires_grad=True)
    x = (H @ W.T) * lmh_oracle.scale_of(T)
    lsm = torch.log_softmax(x, dim=-1)
    tt = torch.tensor(t)
    valid = (tt >= 0) & (tt < V)
    xt = torch.where(valid, x.gather(1, tt.clamp(0, V - 1)[:, None])[:, 0], torch.zeros(N,
                                                                                 dtype=x.dtype))
    lse = torch.logsumexp(x, dim=-1)
    logp = xt - lse
    ent = -(lsm.exp() * lsm).sum(-1)
    loss = (logp * torch.tensor(gl)).sum() + (ent * torch.tensor(ge)).sum() \
        + (lse * torch.tensor(gs)).sum()
    loss.backward()
    np.testing.assert_allclose(dh, H.grad.numpy(), rtol=1e-10, atol=1e-12)
    np.testing.assert_allclose(dw, W.grad.numpy(), rtol=1e-10, atol=1e-12)


def test_vocab_chunk_plan():
    """The chunked head's vocabulary plan (host logic): chunks cover the
    vocabulary in order without gaps; small batches take 32768-column chunks
    with a remainder of at least 16384 + 1024 columns cut into 16384 + the
    rest; larger batches take balanced chunks of a multiple of 1024 columns
    within 128 MiB; an explicit width gives equal chunks and no cut."""
    from kernel_opt import vocab_chunk, vocab_chunks

    def check_cover(plan, V):
        c = 0
        for c0, n in plan:
            assert c0 == c and n >= 1
            c += n
        assert c == V

    qwen = vocab_chunks(1024, 152064)
    check_cover(qwen, 152064)
    assert [n for _, n in qwen] == [32768] * 4 + [16384, 4608]
    assert [n for _, n in vocab_chunks(300, 152064)] == [32768] * 4 + [16384, 4608]
    # a remainder below 16384 + 1024 stays whole; 16384 + 1024 is cut
    assert [n for _, n in vocab_chunks(1024, 32768 + 17407)] == [32768, 17407]
    assert [n for _, n in vocab_chunks(1024, 32768 + 17408)] == [32768, 16384, 1024]
    assert [n for _, n in vocab_chunks(1024, 20000)] == [16384, 3616]
    assert [n for _, n in vocab_chunks(1024, 32768)] == [32768]
    assert [n for _, n in vocab_chunks(5, 300)] == [300]
    # larger batches: balanced, whole multiples of 1024 but the last, <= 128 MiB
    for N, V in ((2048, 152064), (8192, 152064), (4096, 151936), (32768, 262144)):
        plan = vocab_chunks(N, V)
        check_cover(plan, V)
        widths = [n for _, n in plan]
        assert all(w == widths[0] for w in widths[:-1]) and widths[-1] <= widths[0]
        assert widths[0] % 1024 == 0 and N * widths[0] * 2 <= 128 << 20
        assert widths[0] == vocab_chunk(N, V)
    # an explicit width: equal chunks, the last the rest, never cut
    assert [n for _, n in vocab_chunks(1024, 152064, chunk_vocab=20000)] == [20000] * 7 + [12064]
    assert [n for _, n in vocab_chunks(1024, 100, chunk_vocab=1000)] == [100]
    # fp32 halves the columns that fit the small-batch rule
    assert vocab_chunk(1024, 152064, elem_bytes=4) != 32768


@pytest.mark.parametrize("elsewhere", ["hidden", "weight", "targets"])
def test_operands_on_two_devices_are_refused(elsewhere):
    """Refused before any launch, by every entry point of the head: the kernels
    get raw pointers and run on one device's stream.  Shape-only tensors stand
    for those of two GPUs."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    import kernel_opt
    from kernel_opt._head import mfma_operands
    with FakeTensorMode():
        dev = {k: "cuda:1" if k == elsewhere else "cuda:0" for k in ("hidden", "weight", "targets")}
        h = torch.empty(1, 1024, 1024, dtype=torch.bfloat16, device=dev["hidden"])
        w = torch.empty(32000, 1024, dtype=torch.bfloat16, device=dev["weight"])
        t = torch.empty(1, 1024, dtype=torch.int64, device=dev["targets"])
        old = torch.empty(1, 1024, device=dev["hidden"])
        adv = torch.empty(1, device=dev["hidden"])
        for impl in ("chunked", "mfma"):
            with pytest.raises(RuntimeError, match="same device"):
                kernel_opt.fused_linear_logprob_entropy_forward(h, w, t, impl=impl)
            with pytest.raises(RuntimeError, match="same device"):
                kernel_opt.fused_linear_logprob_entropy(h, w, t, impl=impl)
        for level in ("token", "sequence"):
            with pytest.raises(RuntimeError, match="same device"):
                kernel_opt.fused_linear_grpo_step(h, w, t, old, adv, importance_level=level)
        if elsewhere != "targets":
            assert not mfma_operands(h.view(-1, 1024), w)


@pytest.mark.parametrize("n_tokens", [1, 255, 1024, 1025, 2048, 8192, 70000, 300000])
@pytest.mark.parametrize("vocab", [1, 256, 16384, 50257, 152064])
def test_mfma_backward_chunks_cover_the_vocabulary(n_tokens, vocab):
    from kernel_opt.lmhead import MFMA_CHUNK_MAX_BYTES, _mfma_chunks
    plan = _mfma_chunks(n_tokens, vocab, None)
    assert [c0 for c0, _ in plan] == [sum(n for _, n in plan[:i]) for i in range(len(plan))]
    assert sum(n for _, n in plan) == vocab and min(n for _, n in plan) >= 1
    cols = plan[0][1]
    assert cols == vocab or cols % 256 == 0
    # one tile of columns, or within the limit
    assert cols <= 256 or 2 * n_tokens * cols <= MFMA_CHUNK_MAX_BYTES


@pytest.mark.parametrize("n_tokens,chunk_vocab", [(1, None), (4, None), (1, 5000000),
                                                   (2000, 4194303)])
def test_mfma_backward_chunks_stay_within_the_row_stride(n_tokens, chunk_vocab):
    """Millions of columns: every chunk's d_logits rows, padded to 8 columns,
    are within the stride that the products take."""
    from kernel_opt.lmhead import _mfma_chunks
    plan = _mfma_chunks(n_tokens, 9000001, chunk_vocab)
    assert [c0 for c0, _ in plan] == [sum(n for _, n in plan[:i]) for i in range(len(plan))]
    assert sum(n for _, n in plan) == 9000001
    assert max(-(-n // 8) * 8 for _, n in plan) <= (2 ** 31 - 1) // 512


@pytest.mark.parametrize("n_tokens", [7900, 8192, 8300, 16384, 70000, 400000])
@pytest.mark.parametrize("vocab", [5000, 16384, 50257, 152064])
def test_mfma_backward_chunks_of_large_batches_stay_wide(n_tokens, vocab):
    """A chunk of few columns is a short K between two passes over d_hidden's
    accumulator: 8192 columns at least, in whole rounds of the 256 CUs."""
    from kernel_opt.lmhead import _mfma_chunks
    plan = _mfma_chunks(n_tokens, vocab, None)
    cols = plan[0][1]
    assert cols == vocab or 8192 <= cols <= 8192 * 1.25
    assert all(n == cols for _, n in plan[:-1])
    if cols < vocab:
        tiles = cols // 256 * -(-n_tokens // 256)
        assert tiles / (-(-tiles // 256) * 256) > 0.95


def test_large_batches_take_the_faster_products():
    """The measured sides of the rules: logits through the kernels from 7/10
    real tokens up to 4096, d_hidden up to 4096 or over 2^17 columns."""
    from kernel_opt._head import d_hidden_pays, d_weight_pays, logits_pay
    assert logits_pay(1024, 152064, 3584) and logits_pay(4096, 50264, 768)
    assert not logits_pay(8192, 152064, 3584) and not logits_pay(65536, 16384, 1024)
    assert d_hidden_pays(4096, 16384, 1024) and d_hidden_pays(8192, 152064, 3584)
    assert not d_hidden_pays(8192, 32000, 4096) and not d_hidden_pays(65536, 8192, 4096)
    assert d_weight_pays(32000, 4096) and not d_weight_pays(8192, 768)
