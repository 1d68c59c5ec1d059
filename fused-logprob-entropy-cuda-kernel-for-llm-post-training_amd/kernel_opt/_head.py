"""The LM head's products through the hand-written MFMA kernels
(csrc/klp_lmhead.hip, csrc/klp_head_gemm.hip): what the chunked head and the
linear GRPO step run where the operands allow it and the kernels are the
faster ones.

``mfma_operands``: bf16 / fp16, a hidden size that is a multiple of 64,
16-byte aligned rows.  Elsewhere (fp32, odd hidden sizes) the callers keep the
library GEMMs.

``logits_pay`` / ``d_weight_pays`` / ``d_hidden_pays``: small products are one
launch's time in the library, while a 256 x 256 tile a workgroup leaves most
of the chip idle there and d_hidden is two launches.  Ours against the library
(bf16, us, launches queued):
    N     V       D     logits       d_weight     d_hidden
    16    16384   512   15 / 6       10 / 11      29 / 21
    64    16384   512   15 / 6       10 / 9       31 / 68
    64    16384   1024  23 / 9       11 / 12      27 / 81
    128   32000   1024  24 / 15      20 / 23      37 / 101
    256   50240   2048  48 / 57      79 / 104     73 / 207
    512   32000   1024  32 / 36      39 / 45      50 / 146
    64    152064  3584  203 / 204
    192   152064  3584  269 / 287
    320   152064  3584  417 / 423
    320   50240   2048  72 / 72
    320   32000   4096  90 / 75
    320   128256  1024  107 / 101
    512   32000   4096  102 / 98
    512   50240   2048  92 / 101
    1024  152064  3584  843 / 902    971 / 1198   895 / 1475
From 8192 tokens on the library's logits and, for vocabularies (or chunks of
them) below 2^17, its d_hidden are ahead: it reaches 1450-1500 TFLOP/s there, ours
1300-1400, one workgroup a CU whose tile's stores overlap with nothing (65536
tokens of [16384, 1024]: the forward's fold of the same tiles 1740 us, writing
them 2230).  Fewer token blocks at a time on an XCD, for its L2: 8192 tokens of
[50264, 768] 701 -> 591 us, of [152064, 3584] 6623 -> 6285, [16384, 1024] and
[32000, 4096] unchanged; all behind the library still.
    4096  16384   1024  114 / 115    107 / 134    124 / 154
    4096  50264   768   316 / 361    289 / 357    324 / 526
    4096  32000   4096  742 / 723    841 / 1031   840 / 791
    4096  152064  3584  3220 / 3085  3515 / 4076  3643 / 4915
    8192  16384   1024  265 / 215    201 / 252    224 / 263
    8192  50264   768   700 / 581    593 / 657    673 / 590
    8192  32000   4096  1573 / 1494  1668 / 2084  1660 / 1582
    8192  152064  3584  6622 / 6119  7021 / 7971  7152 / 9235
    16384 16384   1024  581 / 422    418 / 525    436 / 415
    16384 128256  2048  6835 / 6316  6793 / 7761  6586 / 6533
    65536 32000   4096  12.6 / 11.6  13.8 / 16.3  13.4 / 13.0 (ms)
The logits' token blocks of 256 (192, 128) do a remainder's work in full: the
library is ahead where fewer than 7/10 of the padded tokens are real ones.
"""
from __future__ import annotations

import torch

from ._library import DTYPE_CODES, check_status, lib, ptr

MAX_LD = (2 ** 31 - 1) // 512  # 32-bit byte offsets within 256 rows


def row_stride(t: torch.Tensor) -> int:
    return t.stride(0) if t.size(0) > 1 else t.size(1)


def _rows_ok(t: torch.Tensor) -> bool:
    ld = row_stride(t)
    return t.data_ptr() % 16 == 0 and ld % 8 == 0 and t.size(1) <= ld <= MAX_LD


def mfma_operands(h2: torch.Tensor, weight: torch.Tensor) -> bool:
    """True when the MFMA kernels take hidden ``[N, D]`` and weight ``[V, D]``
    (one dtype, one device, rows with unit stride)."""
    return (h2.device == weight.device and h2.dtype in (torch.bfloat16, torch.float16)
            and h2.size(0) > 0 and h2.size(1) >= 64 and h2.size(1) % 64 == 0 and h2.stride(1) == 1
            and weight.stride(1) == 1 and _rows_ok(h2) and _rows_ok(weight))


def logits_pay(n_tokens: int, vocab: int, dim: int) -> bool:
    padded = -(-n_tokens // 256) * 256
    return (10 * n_tokens >= 7 * padded and n_tokens * vocab * dim >= 15 << 30
            and n_tokens <= 4096 and vocab % 8 == 0)


def d_weight_pays(vocab: int, dim: int) -> bool:
    return vocab * dim >= 16 << 20


def d_hidden_pays(n_tokens: int, vocab: int, dim: int) -> bool:
    return (n_tokens * vocab * dim >= 1 << 29
            and (n_tokens <= 4096 or vocab >= 1 << 17))


def logits_into(out: torch.Tensor, h2: torch.Tensor, weight: torch.Tensor, stream) -> None:
    """``out[:, :] = h2 @ weight^T``, rounded once to the dtype."""
    check_status(lib.klp_lmh_logits(DTYPE_CODES[h2.dtype], ptr(h2), row_stride(h2), ptr(weight),
                                    row_stride(weight), h2.size(0), weight.size(0), h2.size(1),
                                    ptr(out), row_stride(out), stream))


def d_weight_into(out: torch.Tensor, d: torch.Tensor, ld_d: int, h2: torch.Tensor,
                  stream) -> None:
    """``out = d^T @ h2`` for d_logits ``[N, out.size(0)]`` with row stride
    ``ld_d``."""
    check_status(lib.klp_head_dweight(DTYPE_CODES[h2.dtype], ptr(d), ld_d, h2.size(0), out.size(0),
                                      ptr(h2), row_stride(h2), h2.size(1), ptr(out),
                                      row_stride(out), stream))


def d_hidden_into(out: torch.Tensor | None, acc: torch.Tensor | None, accumulate: bool,
                  d: torch.Tensor, ld_d: int, n_tokens: int, weight: torch.Tensor,
                  stream) -> None:
    """``s = d @ weight`` (+ ``acc`` with ``accumulate``) in float32, into
    ``out`` (rounded once) or, with ``out`` None, into ``acc``."""
    V, D = weight.shape
    nbytes = lib.klp_head_dhidden_workspace_bytes(n_tokens, V, D)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=weight.device)
    check_status(lib.klp_head_dhidden(DTYPE_CODES[weight.dtype], ptr(d), ld_d, n_tokens, V,
                                      ptr(weight), row_stride(weight), D, ptr(acc),
                                      int(accumulate), ptr(out), ptr(ws), nbytes, stream))
