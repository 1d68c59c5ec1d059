// klp_lmhead.hip — fused LM head + per-token logprob / entropy (forward, and
// the backward's d_logits), for gfx950.  The reference names this as its
// natural follow-up (a Liger-style fused linear + loss,
// docs/FINAL_REPORT.md:439-450) and does not build it.
//
//   logits[n, v] = scale * sum_k hidden[n, k] * weight[v, k]      (fp32)
//   logprob[n] = logits[n, t_n] - lse[n],  entropy[n], lse[n]  as klp_fwd
//
// without writing the [N, V] logits anywhere.  hidden is [N, D] and
// weight [V, D], bf16 or fp16 (nn.Linear's layout), both K-contiguous.
//
// klp_lmh_kernel, forward (kFold): one workgroup (4 waves, 2 x 2) per (token block of
// 256, vocab chunk of `tiles_per_chunk` tiles of 256 rows).  Per vocab tile
// it computes the 256 x 256 block of logits^T with v_mfma_f32_16x16x32_bf16,
// each wave a 128 x 128 part of it (64 accumulator blocks, 256 AGPRs).  Where
// that leaves less for the matrix cores to do (few tokens, or a remainder
// block that would be mostly padding) token blocks of 192 or 128, a wave
// 128 x 96 or 128 x 64:
//  - the transposed orientation puts vocab rows on the MFMA's M side, so a
//    lane's accumulators belong to 8 tokens, 32 vocab rows of each: the
//    online softmax update runs lane-locally, with no cross-lane reduction
//    until the end of the chunk;
//  - K advances in stages of 64 columns, a whole 128-byte line of every row,
//    so that no line is asked for in two halves, the second waiting behind
//    the first's pending miss (TCP_PENDING_STALL_CYCLES, 1024 tokens of
//    [152064, 3584]: 1.5e8 a launch, 3.2e8 with 64-byte stages);
//  - the stages go through LDS by direct copies (buffer_load_dwordx4 ... lds,
//    no register staging), all 160 KB of it: a ring of 3 stages of weight
//    rows (32 KB each), which come from HBM, and of 2 stages of hidden rows,
//    which the XCD's L2 holds.  A slot is refilled once every wave has read
//    the stage it held: weight copies have 1.75 stages to land, hidden ones
//    0.75.  The rings run across tile boundaries, and past the last stage
//    the copies go through a descriptor of length 0, which keeps the count
//    of copies in flight, and with it the vmcnt waits, the same on every path;
//  - LDS rows are 128 bytes; the 16-byte chunk index is XOR-swizzled with
//    row bits 1..3 (swz) so that the MFMA operand reads are free of bank
//    conflicts;
//  - operands are read one half stage (32 columns) ahead, two ds_reads per
//    8 MFMAs in source order, and each copy has a slot between two MFMAs;
//    there is one barrier per stage, after the last read of the stage;
//  - after each tile the block's logits are folded into per-lane
//    (m, z, t) states (absorb() of klp_device.h), 32 values of a token at a
//    time; only the tile at the vocabulary's end compares rows, and only
//    tokens whose target lies in the tile look for it.
// At the end of the chunk the four lanes of a token and the two waves of a
// token half merge; the chunk's partial state per token goes to the
// workspace, and a target's logit straight from the lane that holds it.
// klp_lmh_combine_kernel merges the chunks of each token (one wave per token,
// a fixed order) and applies the output formulas.
//
// The backward (kGradient) runs the same tiles and replaces the fold with the
// gradient of klp_bwd, written to d_logits; kLogits writes the logits.
//
// Bound: power.  At 1024 tokens of a [152064, 3584] weight the MFMAs take 4/5
// of the kernel's cycles, and the chip lowers its clock under them: 1.85 GHz,
// against 2.4 GHz with the copies alone or the MFMAs alone (either of which
// takes 550-600 us).  The launch pair takes 800 us (1396 TFLOP/s) end to end,
// where 64-byte stages, 32x32x16 MFMAs and a fold that compared every element
// with the target took 1239.  32x32x16 MFMAs at this tile and ring: 840-848
// us against 797-821 for the main loop alone, at 1.62 against 1.85 GHz.  Up
// to 128 tokens the weight's bytes bound it: 16 tokens 191 us (5.7 TB/s) with
// blocks of 128, 232 with blocks of 256.  257-384 tokens, two blocks of 192:
// 300 tokens 368 us, 432 with blocks of 256, most of the second one padding
// (the library's GEMM per vocabulary chunk, which this kernel replaced: 401).
//
// Workgroup order: workgroup b runs on XCD b % 8 (round-robin dispatch).
// Consecutive workgroups of one XCD take the token blocks of one vocab
// chunk, so the chunk's weight rows are fetched from HBM once per XCD and
// shared through its L2 by the token blocks running there together.
#include "klp_launch.h"
#include "klp_mfma.h"

namespace klp {

namespace {

using namespace mfma;

constexpr int kBV = kTile;  // vocab rows per tile

enum : int { kFold = 0, kGradient = 1, kLogits = 2 };

}  // namespace

// kMode kFold: the forward (partial states per vocab chunk); kGradient: the
// backward's d_logits, the same logits tiles turned into the gradient of
// klp_bwd (grad_one, klp_device.h) and written in DT; kLogits: the logits
// themselves, rounded to DT (kRound, not scaled).  kRound: each logit is
// rounded to DT before it is scaled and used, as a GEMM that writes DT does.
// kTokBlocks: 16-token blocks per wave, 8, 6 or 4 (256, 192 or 128 tokens a
// workgroup).
// kFar: row strides of any size (the others address a block's rows with 32-bit
// offsets): every lane copies from a 64-bit address of its own, and rows past
// the matrix's end are its last one instead of zeros.
template <int DT, int kMode, bool kRound, bool kScaled, int kTokBlocks, bool kFar>
__global__ __launch_bounds__(kThreads) void klp_lmh_kernel(LmhParams p) {
    constexpr int kTokSide = 16 * kTokBlocks;  // a wave's tokens
    constexpr int kBT = 2 * kTokSide;          // the workgroup's
    constexpr int kTokSlot = kBT * kRowBytes;
    constexpr int kTokRing = kASlots * kSlotBytes;  // LDS offset of the hidden rows' ring
    // MFMAs per half stage, and between two of its 8 weight copies.
    constexpr int kSteps = kBlocks * kTokBlocks;
    constexpr int kCopyStep = kSteps / 2 / kCopies;
    // The rings (with 8 token blocks all 160 KB of LDS); the end-of-chunk
    // merge reuses them.
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kTokRing + kBSlots * kTokSlot];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wv = wave & 1;   // vocab half (128 rows) of the tile
    const int wt = wave >> 1;  // token half (128 tokens) of the block

    // Workgroup -> (token block, vocab chunk), XCD-aware (see above).
    const int64_t bid = blockIdx.x;
    const int64_t xcd = bid % 8;
    const int64_t local = bid / 8;
    const int64_t tb = local % p.n_tblocks;
    const int64_t chunk = (local / p.n_tblocks) * 8 + xcd;
    if (chunk >= p.n_chunks) return;  // padding workgroups of the last round

    const int64_t tok0 = tb * kBT;
    const int n_k = static_cast<int>(p.dim / kBK);
    const int64_t tile_first = chunk * p.tiles_per_chunk;
    int64_t tile_end = tile_first + p.tiles_per_chunk;
    if (tile_end > p.n_vtiles) tile_end = p.n_vtiles;

    // Copies.  Lane l of wave w fills, with copy j, chunk l % 8 of slot row
    // 32 j + 8 w + l / 8, which holds global chunk (l % 8) ^ swz(row) of
    // that row (swz reads row bits 1..3, the same for every j).  Rows past
    // the matrix's end lie past the descriptor and read as zeros (their
    // logits are masked or never written).
    const int crow = wave * 8 + (lane >> 3);
    const int cchunk = (lane & 7) ^ swz(crow);
    const uint32_t w_off = static_cast<uint32_t>(crow * p.ld_weight * 2 + cchunk * 16);
    const uint32_t h_off = static_cast<uint32_t>(crow * p.ld_hidden * 2 + cchunk * 16);
    const uint32_t w_step = static_cast<uint32_t>(p.ld_weight * 64);  // 32 rows
    const uint32_t h_step = static_cast<uint32_t>(p.ld_hidden * 64);
    auto rows_rsrc = [](const uint16_t* base, int64_t rows, int64_t ld, int64_t most) {
        return __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint16_t*>(base), 0,
            static_cast<int>((rows < most ? rows : most) * ld * 2), 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t h_rs =
        rows_rsrc(p.hidden + tok0 * p.ld_hidden, p.n_tokens - tok0, p.ld_hidden, kBT);
    auto tile_rsrc = [&](int64_t vt) {
        const bool more = vt < tile_end;
        const int64_t v0 = (more ? vt : tile_first) * kBV;
        return rows_rsrc(p.weight + v0 * p.ld_weight, more ? p.vocab - v0 : 0, p.ld_weight, kBV);
    };
    // The stages to be copied next, and their slots.
    int64_t w_tile = tile_first;
    int w_k = 0, w_slot = 0, h_k = 0, h_slot = 0;
    __amdgpu_buffer_rsrc_t w_rs = tile_rsrc(w_tile);
    // kFar: this lane's 16 bytes of `row` (or of the last row), stage k.
    auto copy_far = [&](const uint16_t* base, int64_t row, int64_t rows, int64_t ld, int k,
                        unsigned char* to) {
        if (row > rows - 1) row = rows - 1;
        __builtin_amdgcn_global_load_lds(base + row * ld + k * kBK + cchunk * 8, (lds_void*)to, 16,
                                         0, 0);
    };
    auto copy_w = [&](int j) {
        unsigned char* to = lds + w_slot * kSlotBytes + (wave + 4 * j) * 1024;
        if constexpr (kFar)
            copy_far(p.weight, w_tile * kBV + 32 * j + crow, p.vocab, p.ld_weight, w_k, to);
        else
            __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rs, (lds_void*)to, 16, w_off,
                                                     j * w_step + w_k * kRowBytes, 0, 0);
        if (j == kCopies - 1) {
            if (++w_k == n_k) {
                w_k = 0;
                w_rs = tile_rsrc(++w_tile);
            }
            w_slot = w_slot == kASlots - 1 ? 0 : w_slot + 1;
        }
    };
    auto copy_h = [&](int j) {
        unsigned char* to = lds + kTokRing + h_slot * kTokSlot + (wave + 4 * j) * 1024;
        if constexpr (kFar)
            copy_far(p.hidden, tok0 + 32 * j + crow, p.n_tokens, p.ld_hidden, h_k, to);
        else
            __builtin_amdgcn_raw_ptr_buffer_load_lds(h_rs, (lds_void*)to, 16, h_off,
                                                     j * h_step + h_k * kRowBytes, 0, 0);
        if (j == kTokBlocks - 1) {
            if (++h_k == n_k) h_k = 0;
            h_slot ^= 1;
        }
    };

    // Operands.  Block i of a side is rows 16 i .. 16 i + 15 of the wave's
    // half; lane l holds row l % 16, K columns 8 (l / 16) .. + 7 of the half
    // stage's 32.
    const int lrow = lane & 15;
    const int lq = lane >> 4;
    const int lf = swz(lrow);
    int rw_slot = 0, rh_slot = 0;  // slots being read
    auto w_src = [&](int half, int i) {
        return *reinterpret_cast<const operand*>(lds + rw_slot * kSlotBytes + wv * (kSlotBytes / 2) +
                                                lrow * kRowBytes +
                                                (((4 * half) ^ (lq ^ lf)) << 4) + i * 16 * kRowBytes);
    };
    auto h_src = [&](int half, int i) {
        return *reinterpret_cast<const operand*>(lds + kTokRing + rh_slot * kTokSlot +
                                                wt * (kTokSlot / 2) + lrow * kRowBytes +
                                                (((4 * half) ^ (lq ^ lf)) << 4) + i * 16 * kRowBytes);
    };

    // The lane's tokens: block b's is tok0 + wt * kTokSide + 16 b + l % 16.
    const int64_t my_tok = tok0 + wt * kTokSide + lrow;
    Stat st[kTokBlocks];
    int my_tgt[kTokBlocks];  // vocab and n_tokens are below 2^31
#pragma unroll
    for (int b = 0; b < kTokBlocks; ++b) {
        st[b] = stat_empty();
        const int64_t tok = my_tok + 16 * b;
        const int64_t t = kMode != kLogits && tok < p.n_tokens ? p.targets[tok] - p.target_offset : -1;
        my_tgt[b] = t >= 0 && t < p.vocab ? static_cast<int>(t) : -1;
    }

    // Prologue: stages 0 and 1.  The steady state's order of copies: hidden
    // of stage g + 2 after the barrier in stage g, weight of stage g + 3 at
    // the start of stage g + 1.
#pragma unroll
    for (int j = 0; j < kCopies; ++j) copy_w(j);
#pragma unroll
    for (int j = 0; j < kTokBlocks; ++j) copy_h(j);
#pragma unroll
    for (int j = 0; j < kCopies; ++j) copy_w(j);
#pragma unroll
    for (int j = 0; j < kTokBlocks; ++j) copy_h(j);
    pin();
    __builtin_amdgcn_s_waitcnt(waitcnt(kCopies + kTokBlocks, 15));
    __builtin_amdgcn_s_barrier();
    pin();
    // Half a stage ahead: all blocks of the token side (two sets, in turn)
    // and blocks 0..3 of the vocab side; its blocks 4..7 are read under the
    // MFMAs of 0..3.
    operand aw[kBlocks], bh[2][kTokBlocks];
#pragma unroll
    for (int i = 0; i < kTokBlocks; ++i) bh[0][i] = h_src(0, i);
#pragma unroll
    for (int i = 0; i < 4; ++i) aw[i] = w_src(0, i);

    for (int64_t vt = tile_first; vt < tile_end; ++vt) {
        f32x4 acc[kBlocks][kTokBlocks];
        // One stage: 2 x kSteps MFMAs, its copies and operand reads placed
        // between them by hand.
        auto stage = [&](auto first_tag) {
            constexpr bool kFirst = decltype(first_tag)::value;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
#pragma unroll
                for (int i = 0; i < kSteps; ++i) {
                    const int a = i / kTokBlocks, b = i % kTokBlocks;
                    if (q == 1 && i == kSteps / 2) {
                        // This wave has read all of the stage, and its copies of
                        // the next one have landed (in flight, at most: the 8
                        // weight copies after those).  After the barrier so for
                        // every wave: the stage's slots are free, the next
                        // stage's are full.
                        pin();
                        __builtin_amdgcn_s_waitcnt(waitcnt(kCopies, 0));
                        __builtin_amdgcn_s_barrier();
                        pin();
                        rw_slot = rw_slot == kASlots - 1 ? 0 : rw_slot + 1;
                        rh_slot ^= 1;
                    }
                    mul_add<DT>(acc[a][b], aw[a], bh[q][b], kFirst && q == 0);
                    if (i < kSteps / 2) {
                        if (b == kTokBlocks / 2 - 1) aw[4 + a] = w_src(q, 4 + a);
                        if (q == 0 && i % kCopyStep == kCopyStep / 2) copy_w(i / kCopyStep);
                    } else {
                        const int n = (i - kSteps / 2) / 4;
                        if (i % 4 == 1) bh[q ^ 1][n] = h_src(q ^ 1, n);
                        if (b == kTokBlocks - 1) aw[a - 4] = w_src(q ^ 1, a - 4);
                        if (q == 1 && i % 4 == 2) copy_h(n);
                    }
                    pin();
                }
            }
        };
        stage(std::true_type{});
        for (int k = 1; k < n_k; ++k) stage(std::false_type{});
        drain();
        pin();

        // Accumulator r of block (a, b) holds tile row
        // wv * 128 + 16 a + 4 (l / 16) + r of the lane's token b.
        const int64_t v0 = vt * kBV;
        const int row0 = wv * kWaveSide + 4 * lq;
        const int64_t left = p.vocab - v0;
        const int vlim = left < kBV ? static_cast<int>(left) : kBV;
        // Values 8 g .. 8 g + 7 of the lane's 32 of token b: rows 16 (2 g) + i
        // and 16 (2 g + 1) + i beyond row0, i = 0..3.
        auto values = [&](int b, int g, float* x) {
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = value(acc[2 * g + j / 4][b][j % 4]);
            if constexpr (kRound) {
#pragma unroll
                for (int j = 0; j < 8; j += 2) round2<DT>(x[j], x[j + 1]);
            }
            if constexpr (kScaled) {
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] *= p.scale;
            }
        };
        if constexpr (kMode != kFold) {
            // Output columns v0 .. of the lane's tokens; lane quarters trade
            // halves so that 16 bytes go out a lane, 64 a token and store.  At
            // the vocabulary's end, or where rows are not 16-byte aligned, 8
            // bytes a lane or single elements, up to column n_out.
            RowGrad rg[kBlocks];
            if constexpr (kMode == kGradient) {
#pragma unroll
                for (int b = 0; b < kTokBlocks; ++b) {
                    const int64_t tok = my_tok + 16 * b;
                    const bool ok = tok < p.n_tokens;
                    rg[b] = ok ? row_grad(p.saved_lse[tok], p.saved_entropy[tok],
                                          p.g_logp ? p.g_logp[tok] : 0.0f,
                                          p.g_ent ? p.g_ent[tok] : 0.0f,
                                          p.g_lse ? p.g_lse[tok] : 0.0f)
                               : row_grad(0.0f, 0.0f, 0.0f, 0.0f, 0.0f);
                }
            }
            const bool whole = vlim == kBV && p.out_align >= 16;
            const int64_t out_left = p.n_out - v0;
            const int olim = out_left < kBV ? static_cast<int>(out_left) : kBV;
#pragma unroll
            for (int b = 0; b < kTokBlocks; ++b) {
                const int64_t tok = my_tok + 16 * b;
                const bool ok = tok < p.n_tokens;
                uint16_t* out = p.out + tok * p.ld_out + v0 + wv * kWaveSide;
                const int target = my_tgt[b] - static_cast<int>(v0) - row0;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    float x[8];
                    values(b, g, x);
                    if constexpr (kMode == kGradient) {
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            x[j] = grad_one(x[j], rg[b]);
                            if (16 * (2 * g + j / 4) + j % 4 == target) x[j] += rg[b].g_logp;
                            if (kScaled) x[j] *= p.scale;
                        }
                    }
                    const uint32_t lo[2] = {pack2<DT>(x[0], x[1]), pack2<DT>(x[2], x[3])};
                    const uint32_t hi[2] = {pack2<DT>(x[4], x[5]), pack2<DT>(x[6], x[7])};
                    if (whole) {
                        const u32x4 w = gather8(lo, hi);
                        if (ok) *reinterpret_cast<u32x4*>(out + 32 * g + 8 * lq) = w;
                    } else if (ok) {
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const int r0 = 32 * g + 16 * h;
                            if (r0 >= olim - row0) continue;
                            uint32_t w[2] = {h ? hi[0] : lo[0], h ? hi[1] : lo[1]};
                            const int n = vlim - row0 - r0;  // of the 4, the vocabulary's
                            if (n < 4) w[1] = n == 3 ? w[1] & 0xFFFFu : 0u;
                            if (n < 2) w[0] = n == 1 ? w[0] & 0xFFFFu : 0u;
                            uint16_t* at = out + r0 + 4 * lq;
                            if (p.out_align >= 8 && olim - row0 - r0 >= 4) {
                                *reinterpret_cast<uint2*>(at) = make_uint2(w[0], w[1]);
                            } else {
#pragma unroll
                                for (int i = 0; i < 4; ++i)
                                    if (i < olim - row0 - r0)
                                        at[i] = static_cast<uint16_t>(w[i / 2] >> (16 * (i & 1)));
                            }
                        }
                    }
                    pin();
                }
            }
            continue;
        }

        // The target logits the lane holds: of every 16 rows from row0, 0..3.
        const int first = static_cast<int>(v0) + row0;
#pragma unroll
        for (int b = 0; b < kTokBlocks; ++b) {
            const int target = my_tgt[b] - first;
            const bool mine = static_cast<uint32_t>(target) < static_cast<uint32_t>(kWaveSide) &&
                              (target & 15) < 4;
            if (__builtin_amdgcn_ballot_w64(mine) == 0) continue;
            float xt = 0.0f;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float x[8];
                values(b, g, x);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (16 * (2 * g + j / 4) + j % 4 == target) xt = x[j];
            }
            if (mine) p.target_logit[my_tok + 16 * b] = xt;
        }
        if (vlim < kBV) {
#pragma unroll
            for (int b = 0; b < kTokBlocks; ++b) {
                // Recomputed per token: the 32 lane masks of the comparisons
                // below would otherwise be kept, and spilled.
                int last = vlim - row0;
                asm volatile("" : "+v"(last));
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    float x[8];
                    values(b, g, x);
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (16 * (2 * g + j / 4) + j % 4 >= last) x[j] = -INFINITY;
                    absorb<8, true>(st[b], x);
                    pin();
                }
            }
        } else {
#pragma unroll
            for (int b = 0; b < kTokBlocks; ++b) {
                const Stat before = st[b];
                float x[32];
#pragma unroll
                for (int g = 0; g < 4; ++g) values(b, g, x + 8 * g);
                absorb<32, false>(st[b], x);
                pin();
                if (needs_clamped_rescan(st[b])) {  // a -inf logit
                    st[b] = before;
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        values(b, g, x);
                        absorb<8, true>(st[b], x);
                    }
                }
            }
        }
    }

    // The last copies (of length 0) write zeros to LDS: before it is reused,
    // or given up.
    __builtin_amdgcn_s_waitcnt(waitcnt(0, 15));
    if constexpr (kMode != kFold) return;

    // Merge the four lanes of each token (vocab rows 4 apart), then the two
    // vocab-half waves of each token half through LDS (the rings' memory:
    // every wave is past its last read of it, and past its last copy into
    // it, once all reach the barrier).
    __syncthreads();
    Stat (*merge_stat)[kBT] = reinterpret_cast<Stat (*)[kBT]>(lds);
#pragma unroll
    for (int b = 0; b < kTokBlocks; ++b) {
        st[b] = combine(st[b], stat_shfl_xor(st[b], 16));
        st[b] = combine(st[b], stat_shfl_xor(st[b], 32));
        if (lane < 16) merge_stat[wv][wt * kTokSide + 16 * b + lane] = st[b];
    }
    __syncthreads();
    const int64_t n = tok0 + tid;
    if (tid < kBT && n < p.n_tokens) {
        const Stat s = combine(merge_stat[0][tid], merge_stat[1][tid]);
        float4* slot = reinterpret_cast<float4*>(p.partials) + chunk * p.n_tokens + n;
        *slot = make_float4(s.m, s.z, s.t, 0.0f);
    }
}

// One wave per token: lane l merges chunks l, l + 64, l + 128, ... in order,
// the lanes then merge in the fixed xor-butterfly order of wave_reduce (so the
// result does not depend on timing), and lane 0 takes the target logit, which
// the lane that met it left in the workspace.
__global__ __launch_bounds__(256) void klp_lmh_combine_kernel(LmhParams p) {
    const int64_t n = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (n >= p.n_tokens) return;
    const float4* part = reinterpret_cast<const float4*>(p.partials);
    Stat acc = stat_empty();
    for (int64_t c = lane; c < p.n_chunks; c += 64) {
        const float4 q = part[c * p.n_tokens + n];
        acc = combine(acc, Stat{q.x, q.y, q.z});
    }
    acc = wave_reduce(acc);
    if (lane != 0) return;
    const int64_t tgt = p.targets[n];
    float x_target = 0.0f;
    if (tgt >= 0 && tgt < p.vocab) x_target = p.target_logit[n];
    const RowOut o = finalize(acc, x_target);
    p.logprob[n] = o.logp;
    p.entropy[n] = o.ent;
    p.lse[n] = o.lse;
}

int64_t lmh_vocab_tiles(int64_t vocab) { return (vocab + kBV - 1) / kBV; }

template <int DT, int kMode, bool kRound, bool kScaled>
static hipError_t launch_lmh_s(const LmhParams& p, hipStream_t stream) {
    // Round the chunk count up to a multiple of 8 (one per XCD per round);
    // padding workgroups exit at once.
    const int64_t chunks8 = (p.n_chunks + 7) / 8 * 8;
    const dim3 grid(static_cast<unsigned>(chunks8 * p.n_tblocks));
    if constexpr (DT == kBF16 && kMode != kLogits && !kRound) {
        if (p.far)
            return launch_kernel(klp_lmh_kernel<DT, kMode, kRound, kScaled, 8, true>, grid,
                                 dim3(kThreads), stream, p);
    }
    if (p.far) return hipErrorInvalidValue;
    if (p.block_tokens == 192)
        return launch_kernel(klp_lmh_kernel<DT, kMode, kRound, kScaled, 6, false>, grid, dim3(kThreads),
                             stream, p);
    if (p.block_tokens == 128)
        return launch_kernel(klp_lmh_kernel<DT, kMode, kRound, kScaled, 4, false>, grid, dim3(kThreads),
                             stream, p);
    return launch_kernel(klp_lmh_kernel<DT, kMode, kRound, kScaled, 8, false>, grid, dim3(kThreads),
                         stream, p);
}

template <int DT, int kMode, bool kRound>
static hipError_t launch_lmh_t(const LmhParams& p, hipStream_t stream) {
    if constexpr (kMode != kLogits) {
        if (p.scale != 1.0f) return launch_lmh_s<DT, kMode, kRound, true>(p, stream);
    }
    return launch_lmh_s<DT, kMode, kRound, false>(p, stream);
}

template <int kMode>
static hipError_t launch_lmh_mode(int dtype, bool rounded, const LmhParams& p,
                                  hipStream_t stream) {
    if (dtype == kFP16 && rounded) return launch_lmh_t<kFP16, kMode, true>(p, stream);
    if (dtype == kBF16 && rounded) return launch_lmh_t<kBF16, kMode, true>(p, stream);
    if constexpr (kMode != kLogits) {
        if (dtype == kBF16) return launch_lmh_t<kBF16, kMode, false>(p, stream);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_lmh_dlogits(int dtype, bool rounded, const LmhParams& p, hipStream_t stream) {
    return launch_lmh_mode<kGradient>(dtype, rounded, p, stream);
}

hipError_t launch_lmh_logits(int dtype, const LmhParams& p, hipStream_t stream) {
    return launch_lmh_mode<kLogits>(dtype, true, p, stream);
}

hipError_t launch_lmh_fwd(int dtype, bool rounded, const LmhParams& p, hipStream_t stream) {
    const hipError_t e = launch_lmh_mode<kFold>(dtype, rounded, p, stream);
    if (e != hipSuccess) return e;
    return launch_kernel(klp_lmh_combine_kernel,
                         dim3(static_cast<unsigned>((p.n_tokens + 3) / 4)), dim3(256), stream, p);
}

}  // namespace klp
