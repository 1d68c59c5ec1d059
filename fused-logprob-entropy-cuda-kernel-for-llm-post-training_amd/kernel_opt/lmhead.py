"""LM head + per-token logprob / entropy without the ``[N, V]`` logits.

``fused_linear_logprob_entropy(hidden, weight, targets)`` returns what
``fused_logprob_entropy(hidden @ weight.T, targets)`` returns, and so does its
backward, while neither pass holds the ``[N, V]`` logits (or their gradient):
the Liger-style head the reference names as its follow-up
(docs/FINAL_REPORT.md:439-450, 490-493) and does not build.

Two implementations:

``impl="chunked"`` (default) rounds each logit once to the input dtype, the
unfused path's numerics.  bf16 / fp16 heads whose hidden size is a multiple of
64 (``_head.mfma_operands``) run the hand-written gfx950 kernels: the forward
is one GEMM with the logprob / entropy reduction as its epilogue
(klp_lmh_fwd_as, csrc/klp_lmhead.hip), and the backward walks the vocabulary
in chunks: per chunk the same GEMM again, with the gradient as its epilogue
(bit-identical logits), then ``d_hidden += d_chunk @ W_chunk`` (fp32) and
``d_weight[chunk] = d_chunk^T @ hidden`` (csrc/klp_head_gemm.hip).  Other heads
walk the vocabulary in chunks in the forward too (:func:`vocab_chunks`): a
library GEMM writes the chunk's logits (``[N, chunk]``, at most 128 MiB) and
``klp_fwd_chunk`` folds them into each token's online state; the last chunk's
launch merges the chunk states in chunk order and writes the outputs.  Their
backward recomputes each chunk with the same GEMM call, applies ``klp_bwd``
with chunk-relative targets, and runs two library GEMMs.

``impl="mfma"`` is the same kernels with the logits kept as fp32 MFMA sums
(never rounded): bf16 inputs, hidden size a multiple of 64.

The backward of either recomputes the logits, one GEMM more than the unfused
path's backward: that is the price of not holding them.  When the loss is
known in the forward, :func:`kernel_opt.fused_linear_grpo_step` computes the
gradients there and needs no recompute.

``fused_linear_logprob_entropy_forward`` is the no-grad entry point (GRPO's
old-policy and reference log-probabilities).
"""
from __future__ import annotations

import torch

from . import _C
from ._head import (MAX_LD, d_hidden_into, d_hidden_pays, d_weight_into, d_weight_pays,
                    mfma_operands)
from ._library import DTYPE_CODES, check_status, device_guard, lib, ptr, stream_handle
from .linear_grpo import _accumulate_f32

__all__ = ["fused_linear_logprob_entropy", "fused_linear_logprob_entropy_forward", "vocab_chunk",
           "vocab_chunks"]


_ptr = ptr


def _check(hidden, weight, targets, impl):
    if impl not in ("chunked", "mfma"):
        raise ValueError(f"impl must be 'chunked' or 'mfma', got {impl!r}")
    if not (hidden.is_cuda and weight.is_cuda and targets.is_cuda):
        raise RuntimeError("hidden, weight and targets must be GPU tensors")
    if not (weight.device == hidden.device and targets.device == hidden.device):
        raise RuntimeError("hidden, weight and targets must be on the same device")
    if impl == "mfma" and (hidden.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16):
        raise RuntimeError("hidden and weight must be bfloat16")
    if hidden.dtype not in DTYPE_CODES or weight.dtype != hidden.dtype:
        raise RuntimeError("hidden and weight must share one dtype: bf16, fp16 or fp32")
    if targets.dtype != torch.int64:
        raise RuntimeError("targets must be int64")
    D = hidden.size(-1)
    if weight.dim() != 2 or weight.size(1) != D:
        raise RuntimeError(f"weight must be [V, {D}], got {tuple(weight.shape)}")
    if tuple(hidden.shape[:-1]) != tuple(targets.shape):
        raise RuntimeError("hidden[..., D] and targets[...] must have the same leading shape")
    if weight.stride(-1) != 1:
        raise RuntimeError("weight rows must have unit stride")
    h2 = hidden.reshape(-1, D)
    if h2.size(0) > 0 and h2.stride(-1) != 1:
        raise RuntimeError("hidden rows must have unit stride")
    return h2, targets.reshape(-1).contiguous()


def _ld(t: torch.Tensor) -> int:
    return t.stride(0) if t.size(0) > 1 else t.size(1)


def _rows_32bit(t: torch.Tensor) -> torch.Tensor:
    """``t``, or its contiguous copy where the products' 32-bit offsets within
    256 rows would not reach (row strides above 4194303 elements)."""
    return t if _ld(t) <= MAX_LD else t.contiguous()


# Vocabulary chunk of the chunked head.  Small batches (a chunk of
# CHUNK_COLS_WIDE columns within CHUNK_WIDE_MAX_BYTES: up to 1024 bf16 tokens)
# take chunks of CHUNK_COLS_WIDE columns, the last one holding the rest.
# Larger batches take about CHUNK_COLS columns, balanced over the vocabulary
# in whole multiples of 1024 (so that no small tail GEMM runs), and fewer
# while one chunk of logits would exceed CHUNK_MAX_BYTES, half of the 256 MB
# Infinity Cache, so that the logprob pass over a chunk reads it from the
# cache.  The library GEMM's speed at the chunk shape dominates, and it does
# not follow the width monotonically.  Measured at Qwen2.5-7B's head in bf16
# while it ran this path, which heads that the MFMA kernels take no longer do
# (V = 152064, D = 3584; forward, forward + backward, ms; two runs):
#   1024 tokens: 32768 columns 0.934-0.940, 4.75-4.76; balanced 15360
#                0.975-0.979, 4.79; unfused 0.927-0.932, 3.84
#   2048 tokens: balanced 15360 1.75-1.76, 8.40-8.44; 16384 1.70-1.71,
#                9.80-9.82 (its backward GEMMs are slow); unfused 1.70, 7.04
#   4096 tokens: balanced 15360 3.34, 15.22-15.24; 8192 3.30-3.31,
#                15.30-15.31; unfused 3.25-3.27, 12.94
#   8192 tokens: balanced 8192 6.39-6.40, 30.40-30.46; unfused 6.41-6.43, 24.65
# The forward and the backward use the same chunks: the backward recomputes
# each chunk's logits with the same GEMM call, hence the same values.
# In the small-batch regime a last chunk wider than CHUNK_COLS_WIDE / 2 is
# cut into CHUNK_COLS_WIDE / 2 columns plus the rest: the library GEMM runs
# widths of 16384 and 32768 columns at 5.0-5.1 us per 1024 columns (1024
# tokens, D = 3584), but 18432-22528 at 6.2-6.8 us (V = 152064's remainder of
# 20992: 138.8 us, against 83.4 + ~36 us as 16384 + 4608).  Qwen2.5-7B's head
# at 1024 tokens, forward, one box, launches queued (host-issued): chunks
# 4 x 32768 + 20992 950.3 (927.2) us, 4 x 32768 + 16384 + 4608 942.4
# (908.4) us, unfused 957.7 (923.2) us.
CHUNK_COLS_WIDE = 32768
CHUNK_WIDE_MAX_BYTES = 64 << 20
CHUNK_COLS = 16384
CHUNK_MAX_BYTES = 128 << 20


def vocab_chunk(n_tokens: int, vocab: int, elem_bytes: int = 2,
                chunk_vocab: int | None = None) -> int:
    """Columns per chunk of the chunked head (the last chunk may hold
    fewer)."""
    if chunk_vocab is not None:
        if chunk_vocab < 1:
            raise ValueError(f"chunk_vocab must be >= 1, got {chunk_vocab}")
        return min(int(chunk_vocab), max(vocab, 1))
    if n_tokens * CHUNK_COLS_WIDE * elem_bytes <= CHUNK_WIDE_MAX_BYTES:
        return min(vocab, CHUNK_COLS_WIDE)
    cols = CHUNK_COLS
    while cols > 1024 and n_tokens * cols * elem_bytes > CHUNK_MAX_BYTES:
        cols //= 2
    n_chunks = max(1, -(-vocab // cols))
    per = -(-vocab // n_chunks)
    return min(vocab, -(-per // 1024) * 1024)


def vocab_chunks(n_tokens: int, vocab: int, elem_bytes: int = 2,
                 chunk_vocab: int | None = None) -> list:
    """``(first column, width)`` of every vocabulary chunk of the chunked
    head, in order: chunks of :func:`vocab_chunk` columns, the last one the
    rest; in the small-batch regime a rest of at least half a chunk plus 1024
    columns is cut in two (``CHUNK_COLS_WIDE // 2`` columns, then the
    remainder).  The forward and the backward use the same chunks."""
    vc = vocab_chunk(n_tokens, vocab, elem_bytes, chunk_vocab)
    plan = [(c0, min(vc, vocab - c0)) for c0 in range(0, vocab, vc)]
    wide = n_tokens * CHUNK_COLS_WIDE * elem_bytes <= CHUNK_WIDE_MAX_BYTES
    half = CHUNK_COLS_WIDE // 2
    if chunk_vocab is None and wide and plan and half + 1024 <= plan[-1][1] < CHUNK_COLS_WIDE:
        c0, n = plan[-1]
        plan[-1:] = [(c0, half), (c0 + half, n - half)]
    return plan


# Chunk of d_logits of the MFMA backward, in whole 256-column tiles.  Up to
# 1024 tokens equal chunks within 64 MiB.  Above, 128 MiB: fewer chunks make
# d_hidden's K longer and the passes over its float32 accumulator fewer, and
# their 256 x 256 tiles are a whole number of rounds of the 256 CUs, as nearly
# as they fit, the last chunk holding the rest.  Forward + backward, ms, equal
# chunks within 64 MiB / whole rounds within 128 MiB:
#   [152064, 3584]   700 tokens  2.81-2.88 / 3.00-3.03   1024  3.78-3.79 / 3.81-3.82
#                   1500         5.72-5.76 / 5.53-5.54   2048  7.51-7.53 / 7.20
#                   4096       14.21-14.32 / 14.04-14.08 8192  34.7 / 29.1
#   [100000, 1024]  2000         1.90 / 1.62-1.63
#   [50240, 2048]   2048         1.59 / 1.47             1024  0.87-0.88 / 0.85-0.86
# From about 8192 tokens on, 128 MiB are fewer than 8192 columns: each chunk
# moves the accumulator and its slab (16 bytes a value of d_hidden) for a K that
# shrinks as the batch grows.  A chunk then has about 8192 columns, in whole
# rounds, whatever their bytes up to 8 GiB.  Forward + backward, ms, 128 MiB /
# 8192 columns (in brackets the library path's chunks of 1024-4096 columns):
#   [152064, 3584]  16384 tokens 67 / 58.6 [63]   65536  399-407 / 235 [291]
#   [32000, 4096]  131072       326 / 110 [136]
#   [50257, 768]   131072       146 / 40.7 [79]  400000  754 / 126 [205]
# A chunk's columns are the row stride of its d_logits, which the products
# address with 32-bit offsets: few tokens of millions of columns take several.
MFMA_CHUNK_MAX_COLS = MAX_LD // 256 * 256
MFMA_CHUNK_TOKENS = 1024
MFMA_CHUNK_BYTES = 64 << 20
MFMA_CHUNK_ROUNDS_BYTES = 128 << 20
MFMA_CHUNK_MIN_TILES = 32
MFMA_CHUNK_MAX_BYTES = 8 << 30


def _mfma_chunks(n_tokens: int, vocab: int, chunk_vocab: int | None) -> list:
    """``(first column, width)`` of every chunk of the MFMA backward."""
    if chunk_vocab is not None:
        return vocab_chunks(n_tokens, vocab, 2, min(chunk_vocab, MFMA_CHUNK_MAX_COLS))
    if n_tokens <= MFMA_CHUNK_TOKENS:
        n_chunks = max(1, -(-(n_tokens * vocab * 2) // MFMA_CHUNK_BYTES))
        cols = -(-(-(-vocab // n_chunks)) // 256) * 256
    else:
        tile_bytes = 2 * n_tokens * 256
        tiles = MFMA_CHUNK_ROUNDS_BYTES // tile_bytes
        if tiles * 256 < vocab:
            token_blocks = -(-n_tokens // 256)
            tiles = tiles * token_blocks // 256 * 256 // token_blocks
            if tiles < MFMA_CHUNK_MIN_TILES:
                tiles = -(-MFMA_CHUNK_MIN_TILES * token_blocks // 256) * 256 // token_blocks
            tiles = max(1, min(tiles, MFMA_CHUNK_MAX_BYTES // tile_bytes))
        cols = tiles * 256
    cols = min(cols, MFMA_CHUNK_MAX_COLS)
    return [(c0, min(cols, vocab - c0)) for c0 in range(0, vocab, cols)]


def _chunk_logits(buf, h2, weight, c0, n):
    """logits[:, c0:c0+n] = h2 @ weight[c0:c0+n]^T into a contiguous view of
    ``buf`` through the library: the same call, hence the same values, in the
    forward and the backward of heads without MFMA kernels."""
    out = buf[: h2.size(0) * n].view(h2.size(0), n)
    torch.mm(h2, weight[c0:c0 + n].t(), out=out)
    return out


def _forward_mfma(h2, weight, t, T, rounded, out):
    """The one-GEMM forward; logits rounded to the dtype, or kept in fp32."""
    dev = h2.device
    N, V, D = h2.size(0), weight.size(0), h2.size(1)
    with device_guard(dev.index):
        stream = stream_handle(dev.index)
        # From the allocator on every call: a captured call's then belongs to
        # its graph, and no later call can replace it under a replay.
        ws = torch.empty(lib.klp_lmh_workspace_bytes(N, V, D), dtype=torch.uint8, device=dev)
        check_status(lib.klp_lmh_fwd_as(DTYPE_CODES[h2.dtype], int(rounded), _ptr(h2), _ld(h2),
                                        _ptr(weight), _ld(weight), N, V, D, _ptr(t), T,
                                        _ptr(out[0]), _ptr(out[1]), _ptr(out[2]), _ptr(ws),
                                        ws.numel(), stream))


def _forward_chunked(h2, weight, t, T, plan, out):
    N = h2.size(0)
    n_chunks = len(plan)
    dev = h2.device
    states = torch.empty(n_chunks, N, 4, dtype=torch.float32, device=dev)
    buf = torch.empty(N * max(n for _, n in plan), dtype=h2.dtype, device=dev)
    code = DTYPE_CODES[h2.dtype]
    with device_guard(dev.index):
        stream = stream_handle(dev.index)
        for c, (c0, n) in enumerate(plan):
            lg = _chunk_logits(buf, h2, weight, c0, n)
            check_status(lib.klp_fwd_chunk(_ptr(lg), code, N, n, *_C.row_layout(lg), _ptr(t),
                                           c0, T, _ptr(states), c, n_chunks, _ptr(out[0]),
                                           _ptr(out[1]), _ptr(out[2]), stream))


def _backward_mfma(h2, weight, t, T, plan, lse, ent, gl, ge, gs, need_h, need_w, rounded):
    """d_hidden (float32 or the operands' dtype, or None) and d_weight (their
    dtype, or None), one vocabulary chunk of ``plan`` at a time: d_logits
    exist for one chunk only."""
    N, D, V = h2.size(0), h2.size(1), weight.size(0)
    dev = h2.device
    code = DTYPE_CODES[h2.dtype]
    cols = max(n for _, n in plan)
    own_dh, own_dw = d_hidden_pays(N, cols, D), d_weight_pays(cols, D)
    dh = torch.empty(N, D, dtype=h2.dtype, device=dev) if need_h and own_dh else None
    acc = None
    if need_h and not own_dh:
        acc = torch.zeros(N, D, dtype=torch.float32, device=dev)
    elif need_h and len(plan) > 1:
        acc = torch.empty(N, D, dtype=torch.float32, device=dev)
    dw = torch.empty(V, D, dtype=weight.dtype, device=dev) if need_w else None
    d = torch.empty(N * (-(-cols // 8) * 8), dtype=h2.dtype, device=dev)
    with device_guard(dev.index):
        stream = stream_handle(dev.index)
        for c, (c0, n) in enumerate(plan):
            ld_d = -(-n // 8) * 8
            w_c = weight[c0:c0 + n]
            check_status(lib.klp_lmh_bwd_logits_as(
                code, int(rounded), _ptr(h2), _ld(h2), _ptr(w_c), _ld(weight), N, n, D, _ptr(t),
                c0, T, _ptr(lse), _ptr(ent), _ptr(gl), _ptr(ge), _ptr(gs), _ptr(d), ld_d, stream))
            d_c = d[: N * ld_d].view(N, ld_d)[:, :n]
            if need_h and own_dh:
                d_hidden_into(dh if c == len(plan) - 1 else None, acc, c > 0, d, ld_d, N, w_c,
                              stream)
            elif need_h:
                _accumulate_f32(acc, d_c, w_c)
            if need_w and own_dw:
                d_weight_into(dw[c0:c0 + n], d, ld_d, h2, stream)
            elif need_w:
                torch.mm(d_c.t(), h2, out=dw[c0:c0 + n])
    return acc if need_h and not own_dh else dh, dw


def _backward_chunked(h2, weight, t, T, plan, lse, ent, gl, ge, gs, need_h, need_w):
    """d_hidden (fp32, or None) and d_weight (weight dtype, or None) through
    library GEMMs, one vocabulary chunk of ``plan`` at a time."""
    N, D, V = h2.size(0), h2.size(1), weight.size(0)
    dev = h2.device
    dh = torch.zeros(N, D, dtype=torch.float32, device=dev) if need_h else None
    dw = torch.empty(V, D, dtype=weight.dtype, device=dev) if need_w else None
    cols = max(n for _, n in plan)
    d_buf = torch.empty(N * cols, dtype=weight.dtype, device=dev)
    lg_buf = torch.empty(N * cols, dtype=h2.dtype, device=dev)
    with device_guard(dev.index):
        stream = stream_handle(dev.index)
        for c0, n in plan:
            tc = t - c0  # chunk-relative: a target outside the chunk adds no one-hot term
            lg = _chunk_logits(lg_buf, h2, weight, c0, n)
            d = d_buf[: N * n].view(N, n)
            check_status(lib.klp_bwd_temp(_ptr(lg), DTYPE_CODES[lg.dtype], N, n,
                                          *_C.row_layout(lg),
                                          _ptr(tc), T, _ptr(lse), _ptr(ent), _ptr(gl),
                                          _ptr(ge), _ptr(gs), _ptr(d), stream))
            w_c = weight[c0:c0 + n]
            if need_h:
                _accumulate_f32(dh, d, w_c)
            if need_w:
                torch.mm(d.t(), h2, out=dw[c0:c0 + n])
    return dh, dw


class _FusedLinearLogprobEntropy(torch.autograd.Function):

    @staticmethod
    def forward(ctx, hidden, weight, targets, temperature, impl, chunk_vocab):
        outs = fused_linear_logprob_entropy_forward(hidden, weight, targets, temperature,
                                                    impl=impl, chunk_vocab=chunk_vocab)
        ctx.save_for_backward(hidden, weight, targets, outs[2], outs[1])
        ctx.temperature = temperature
        ctx.impl = impl
        ctx.chunk_vocab = chunk_vocab
        ctx.set_materialize_grads(False)
        return outs

    @staticmethod
    def backward(ctx, g_logp, g_ent, g_lse):
        hidden, weight, targets, lse, ent = ctx.saved_tensors
        need_h, need_w = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        none = (None,) * 4
        if not (need_h or need_w):
            return (None, None) + none
        h2, t = _check(hidden, weight, targets, ctx.impl)
        N, V = h2.size(0), weight.size(0)
        if N == 0:
            return (torch.zeros_like(hidden) if need_h else None,
                    torch.zeros_like(weight) if need_w else None) + none

        def prep(g):
            return None if g is None else g.to(torch.float32, copy=False).reshape(-1).contiguous()

        T = 1.0 if ctx.temperature is None else float(ctx.temperature)
        args = (lse.reshape(-1), ent.reshape(-1), prep(g_logp), prep(g_ent), prep(g_lse), need_h,
                need_w)
        if ctx.impl == "mfma":
            h2, weight = _rows_32bit(h2), _rows_32bit(weight)
        if ctx.impl == "mfma" or mfma_operands(h2, weight):
            dh, dw = _backward_mfma(h2, weight, t, T, _mfma_chunks(N, V, ctx.chunk_vocab), *args,
                                    ctx.impl == "chunked")
        else:
            dh, dw = _backward_chunked(h2, weight, t, T,
                                       vocab_chunks(N, V, h2.element_size(), ctx.chunk_vocab),
                                       *args)
        if dh is not None:
            dh = dh.to(hidden.dtype).reshape(hidden.shape)
        return (dh, dw) + none


def fused_linear_logprob_entropy(hidden: torch.Tensor, weight: torch.Tensor,
                                 targets: torch.Tensor, temperature: float | None = None, *,
                                 impl: str = "chunked", chunk_vocab: int | None = None):
    """Autograd-aware LM head + logprob / entropy: gradients flow to
    ``hidden`` and ``weight`` (see :func:`fused_linear_logprob_entropy_forward`
    for the arguments and the module docstring for the backward)."""
    return _FusedLinearLogprobEntropy.apply(hidden, weight, targets, temperature, impl,
                                            chunk_vocab)


def fused_linear_logprob_entropy_forward(hidden: torch.Tensor, weight: torch.Tensor,
                                         targets: torch.Tensor,
                                         temperature: float | None = None, *,
                                         impl: str = "chunked",
                                         chunk_vocab: int | None = None):
    """Args:
        hidden: ``[..., D]`` on the GPU, rows with unit stride (the leading
            dims must flatten to one stride).
        weight: ``[V, D]`` (an ``nn.Linear`` weight) of hidden's dtype, rows
            with unit stride.
        targets: ``[...]`` int64, same leading shape as ``hidden``.
        temperature: optional T > 0; logits are multiplied by fp32(1/T).
        impl: ``"chunked"`` (bf16 / fp16 / fp32) or ``"mfma"`` (bf16, D a
            multiple of 64, both row strides multiples of 8).
        chunk_vocab: columns per vocabulary chunk where a pass walks the
            vocabulary in chunks (the backward; the forward of heads without
            MFMA kernels); default :func:`vocab_chunks`, or, with them, chunks
            of d_logits of 64 MiB up to 1024 tokens, 128 MiB above and 8192
            columns from about 8192 tokens on.

    Returns ``(logprob, entropy, lse)``, float32, shaped like ``targets``.
    """
    h2, t = _check(hidden, weight, targets, impl)
    D = h2.size(1)
    N, V = h2.size(0), weight.size(0)
    out = [torch.empty(targets.shape, dtype=torch.float32, device=hidden.device)
           for _ in range(3)]
    if N == 0:
        return tuple(out)
    T = 1.0 if temperature is None else float(temperature)
    if not (T > 0.0 and T != float("inf")):
        raise RuntimeError(f"temperature must be finite and > 0, got {T}")
    if impl == "mfma":
        _forward_mfma(h2, weight, t, T, False, out)
    elif mfma_operands(h2, weight):
        if chunk_vocab is not None and chunk_vocab < 1:
            raise ValueError(f"chunk_vocab must be >= 1, got {chunk_vocab}")
        _forward_mfma(h2, weight, t, T, True, out)
    else:
        _forward_chunked(h2, weight, t, T, vocab_chunks(N, V, h2.element_size(), chunk_vocab),
                         out)
    return tuple(out)
