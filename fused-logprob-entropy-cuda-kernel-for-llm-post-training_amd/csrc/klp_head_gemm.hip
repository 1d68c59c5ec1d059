// klp_head_gemm.hip — the two products of the LM head's backward, for gfx950:
//
//   d_weight[v, d] = sum_n d_logits[n, v] * hidden[n, d]     (16-bit out)
//   d_hidden[n, d] = sum_v d_logits[n, v] * weight[v, d]     (float32 sums,
//                    added to an accumulator or rounded once to 16 bits)
//
// of bf16 or fp16 matrices with float32 MFMA sums.  One workgroup (4 waves,
// 2 x 2) computes 256 x 256 tiles of the output, d along the MFMA's M side so
// that a lane holds consecutive d of one output row; the stages, rings,
// copies and their waits are klp_lmh_kernel's (klp_lmhead.hip).
//
// The M side's matrix (hidden, weight) has its K dimension as rows, so has
// d_logits in the d_weight product: these go to LDS as they lie in memory
// (64 K rows of 512 bytes a stage) and are transposed by the operand reads
// (ds_read_b64_tr_b16).  d_logits in the d_hidden product is K-contiguous.
//
// d_weight: K is the token count, a few stages a tile, so a workgroup takes
// several tiles and runs its rings across them.  d_hidden: few tiles with a K
// of the whole vocabulary (chunk); K is split over workgroups, each writes its
// float32 tile to a slab of the workspace, and klp_head_sum_kernel adds the
// slabs in order (the result does not depend on timing).
//
// Workgroup order: workgroup b runs on XCD b % 8; each XCD takes one
// contiguous range of tiles, its 32 workgroups 32 neighbours at a time: up to
// 6 row blocks by 5 or more d tiles, so that a stage's rows are fetched into
// the XCD's L2 once for 5-6 workgroups on either side.
//
// Bound: power and, in d_weight, the output's 1.1 GB and short tiles.  1024
// tokens of a bf16 [152064, 3584] head: d_weight 971 us (1150 TFLOP/s; the
// library GEMM 1198 us), d_hidden 895 us with the sum (1248 TFLOP/s; the
// library 1475 us).  d_weight with 7 consecutive d tiles of one row block a workgroup,
// and the short ring for d_logits: 1140 us, its MFMAs busy half of the time.
#include "klp_launch.h"
#include "klp_mfma.h"

namespace klp {

namespace {

using namespace mfma;

}  // namespace

// kBRows: the N side's matrix has K as rows (d_weight); otherwise it is
// K-contiguous (d_hidden).  kSlab: float32 tiles into slab `split` of the
// workspace; otherwise 16-bit output.
template <int DT, bool kBRows, bool kSlab>
__global__ __launch_bounds__(kThreads) void klp_head_gemm_kernel(HeadGemmParams p) {
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kLdsBytes];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1;   // half of the tile's d
    const int wn = wave >> 1;  // half of the tile's output rows
    // d_logits come from memory (d_weight), or the weight does (d_hidden):
    // that operand takes the long ring, and its copies more time to land.
    constexpr int kARing = kBRows ? 2 : 3;
    constexpr int kBRing = kBRows ? 3 : 2;

    // Workgroup -> every 32nd (workgroups per XCD) item of its XCD's range.
    const int stride = static_cast<int>(gridDim.x / 8);
    const int xcd_items = static_cast<int>((p.n_items + 7) / 8);
    const int xcd = static_cast<int>(blockIdx.x % 8);
    const int item_first = xcd * xcd_items + static_cast<int>(blockIdx.x / 8);
    int item_end = (xcd + 1) * xcd_items;
    if (item_end > p.n_items) item_end = static_cast<int>(p.n_items);
    if (item_first >= item_end) return;

    // An item's place: splits outermost, then groups of p.group row blocks,
    // in each the row blocks fastest, then the d tiles.
    struct Place {
        int m, n, split;
    };
    auto place_of = [&](int item) {
        const uint32_t i = static_cast<uint32_t>(item);
        const uint32_t m_tiles = static_cast<uint32_t>(p.m_tiles);
        const uint32_t n_tiles = static_cast<uint32_t>(p.n_tiles);
        const uint32_t group = static_cast<uint32_t>(p.group);
        const uint32_t split = i / (m_tiles * n_tiles);
        const uint32_t r = i - split * (m_tiles * n_tiles);
        const uint32_t g = r / (group * m_tiles);
        const uint32_t q = r - g * (group * m_tiles);
        const uint32_t left = n_tiles - g * group;
        const uint32_t size = left < group ? left : group;
        const uint32_t m = q / size;
        return Place{static_cast<int>(m), static_cast<int>(g * group + q - m * size),
                     static_cast<int>(split)};
    };
    auto k_first = [&](const Place& t) { return static_cast<int64_t>(t.split) * p.k_per_split; };
    auto k_count = [&](const Place& t) {
        const int64_t left = p.k - k_first(t);
        return static_cast<int>(left < p.k_per_split ? left : p.k_per_split);
    };

    // Copies of K rows: lane l of wave w fills, with copy j, 16-byte chunk
    // l % 32 of slot row k = 8 j + 2 w + l / 32; that chunk holds half
    // (l % 32) / 16, sub-chunk l % 2 of block ((l % 16) / 2) ^ swz_k(k), whose
    // bit 2 is j's bit 0.
    const int krow = 2 * wave + (lane >> 5);
    const int kcol = ((lane & 16) << 3) + (((((lane & 15) >> 1) ^ (krow & 3)) << 4)) +
                     ((lane & 1) << 3);
    // Copies of K-contiguous rows: chunk l % 8 of slot row 32 j + 8 w + l / 8.
    const int crow = wave * 8 + (lane >> 3);
    const int cchunk = (lane & 7) ^ swz(crow);

    constexpr uint32_t kNowhere = 0x80000000u;  // past every descriptor
    const uint32_t a_off[2] = {static_cast<uint32_t>((krow * p.ld_a + kcol) * 2),
                               static_cast<uint32_t>((krow * p.ld_a + (kcol ^ 64)) * 2)};
    const uint32_t a_step = static_cast<uint32_t>(p.ld_a * 16);  // 8 rows
    const uint32_t b_off[2] = {
        static_cast<uint32_t>(kBRows ? (krow * p.ld_b + kcol) * 2 : crow * p.ld_b * 2 + cchunk * 16),
        static_cast<uint32_t>(kBRows ? (krow * p.ld_b + (kcol ^ 64)) * 2 : 0)};
    const uint32_t b_step = static_cast<uint32_t>(kBRows ? p.ld_b * 16 : p.ld_b * 64);

    // The stages to be copied next (their item and the K left in it), and
    // their slots.  Past the last item the descriptors have length 0, which
    // keeps the count of copies in flight the same on every path.
    int a_item = item_first, b_item = item_first;
    int a_slot = 0, b_slot = 0, a_left = 0, b_left = 0, b_rows = 0;
    const uint16_t* a_ptr = p.a;
    const uint16_t* b_ptr = p.b;
    u32x4 a_rs, b_rs;
    // Each descriptor ends with its last row's last column (rounded up to 8):
    // chunks past the matrix within earlier rows read their neighbours, whose
    // outputs are not stored.
    auto rsrc = [](const uint16_t* base, int rows, int64_t ld, int64_t width) {
        return bytes_rsrc(base, rows > 0 ? static_cast<uint32_t>(((rows - 1) * ld + width) * 2) : 0u);
    };
    int64_t a_width = 0, b_width = 0;
    auto a_stage = [&]() { a_rs = rsrc(a_ptr, a_left < kBK ? a_left : kBK, p.ld_a, a_width); };
    auto b_stage = [&]() {
        if constexpr (kBRows) b_rs = rsrc(b_ptr, b_left < kBK ? b_left : kBK, p.ld_b, b_width);
        else b_rs = rsrc(b_ptr, b_left > 0 ? b_rows : 0, p.ld_b, (b_left + 7) & ~7);
    };
    auto a_open = [&]() {
        a_left = 0;
        if (a_item >= item_end) return;
        const Place at = place_of(a_item);
        a_left = k_count(at);
        const int64_t m0 = static_cast<int64_t>(at.m) * kTile;
        a_width = p.m - m0 < kTile ? p.m - m0 : kTile;
        a_ptr = p.a + k_first(at) * p.ld_a + m0;
    };
    auto b_open = [&]() {
        b_left = 0;
        if (b_item >= item_end) return;
        const Place at = place_of(b_item);
        b_left = k_count(at);
        const int64_t n0 = static_cast<int64_t>(at.n) * kTile;
        b_rows = static_cast<int>(p.n - n0 < kTile ? p.n - n0 : kTile);
        b_width = (b_rows + 7) & ~7;
        b_ptr = kBRows ? p.b + k_first(at) * p.ld_b + n0 : p.b + n0 * p.ld_b + k_first(at);
    };
    a_open();
    b_open();
    a_stage();
    b_stage();
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void*)lds));
    auto copy_a = [&](int j) {
        copy_to_lds(a_rs, lds0 + a_slot * kSlotBytes + (wave + 4 * j) * 1024, a_off[j & 1],
                    j * a_step);
        if (j < kCopies - 1) return;
        a_left -= kBK;
        a_ptr += kBK * p.ld_a;
        if (a_left <= 0) {
            a_item += stride;
            a_open();
        }
        a_stage();
        a_slot = a_slot == kARing - 1 ? 0 : a_slot + 1;
    };
    auto copy_b = [&](int j) {
        uint32_t off = b_off[kBRows ? j & 1 : 0];
        // The K-contiguous stage at K's end: chunks past it read as zeros.
        if (!kBRows && b_left < kBK) off = cchunk * 8 < b_left ? off : kNowhere;
        copy_to_lds(b_rs, lds0 + (kARing + b_slot) * kSlotBytes + (wave + 4 * j) * 1024, off,
                    j * b_step);
        if (j < kCopies - 1) return;
        b_left -= kBK;
        b_ptr += kBRows ? kBK * p.ld_b : kBK;
        if (b_left <= 0) {
            b_item += stride;
            b_open();
        }
        b_stage();
        b_slot = b_slot == kBRing - 1 ? 0 : b_slot + 1;
    };
    auto copy_long = [&](int j) { kBRows ? copy_b(j) : copy_a(j); };
    auto copy_short = [&](int j) { kBRows ? copy_a(j) : copy_b(j); };

    // Operands.  Lane l holds row (column of the tile) l % 16 of block i, K
    // values 8 (l / 16) .. + 7 of the half stage's 32.
    const int lrow = lane & 15;
    const int lq = lane >> 4;
    const int lf = swz(lrow);
    const int tr_row = (8 * lq + (lrow >> 2)) * 512 + (lane & 3) * 8;
    const int tr_swz = (lrow >> 2) | ((lq & 1) << 2);
    int ra_slot = 0, rb_slot = 0;  // slots being read
    auto read_rows = [&](int at, int half_tile, int half, int i) {
        const unsigned char* s =
            lds + at + half_tile * 256 + tr_row + ((i ^ tr_swz) << 5) + half * 32 * 512;
        const s16x4 lo = read_tr(s), hi = read_tr(s + 4 * 512);
        return __builtin_bit_cast(
            operand, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    auto a_src = [&](int half, int i) {
        return read_rows(ra_slot * kSlotBytes, wm, half, i);
    };
    auto b_src = [&](int half, int i) {
        const int at = (kARing + rb_slot) * kSlotBytes;
        if constexpr (kBRows) return read_rows(at, wn, half, i);
        else return *reinterpret_cast<const operand*>(
                lds + at + wn * (kSlotBytes / 2) + lrow * kRowBytes +
                (((4 * half) ^ (lq ^ lf)) << 4) + i * 16 * kRowBytes);
    };

    // Prologue: stages 0 and 1.  The steady state's order of copies: the
    // short ring's of stage g + 2 after the barrier in stage g, the long
    // ring's of stage g + 3 at the start of stage g + 1.
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int j = 0; j < kCopies; ++j) copy_long(j);
#pragma unroll
        for (int j = 0; j < kCopies; ++j) copy_short(j);
    }
    pin();
    __builtin_amdgcn_s_waitcnt(waitcnt(2 * kCopies, 15));
    __builtin_amdgcn_s_barrier();
    pin();
    operand av[kBlocks], bv[2][kBlocks];
#pragma unroll
    for (int i = 0; i < kBlocks; ++i) bv[0][i] = b_src(0, i);
#pragma unroll
    for (int i = 0; i < 4; ++i) av[i] = a_src(0, i);

    for (int item = item_first; item < item_end; item += stride) {
        const Place place = place_of(item);
        const int n_k = (k_count(place) + kBK - 1) / kBK;
        f32x4 acc[kBlocks][kBlocks];
        auto stage = [&](auto first_tag) {
            constexpr bool kFirst = decltype(first_tag)::value;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
#pragma unroll
                for (int i = 0; i < 64; ++i) {
                    const int a = i >> 3, b = i & 7;
                    if (q == 1 && i == 32) {
                        // This wave has read all of the stage, and its copies of
                        // the next one have landed; after the barrier so for
                        // every wave.
                        pin();
                        __builtin_amdgcn_s_waitcnt(waitcnt(kCopies, 0));
                        __builtin_amdgcn_s_barrier();
                        pin();
                        ra_slot = ra_slot == kARing - 1 ? 0 : ra_slot + 1;
                        rb_slot = rb_slot == kBRing - 1 ? 0 : rb_slot + 1;
                    }
                    mul_add<DT>(acc[a][b], av[a], bv[q][b], kFirst && q == 0);
                    if (i < 32) {
                        if ((i & 7) == 3) av[4 + a] = a_src(q, 4 + a);
                        if (q == 0 && (i & 3) == 2) copy_long(i >> 2);
                    } else {
                        if ((i & 3) == 1) bv[q ^ 1][(i - 32) >> 2] = b_src(q ^ 1, (i - 32) >> 2);
                        if ((i & 7) == 7) av[a - 4] = a_src(q ^ 1, a - 4);
                        if (q == 1 && (i & 3) == 2) copy_short((i - 32) >> 2);
                    }
                    pin();
                }
            }
        };
        stage(std::true_type{});
        for (int k = 1; k < n_k; ++k) stage(std::false_type{});
        drain();
        pin();

        // Accumulator r of block (a, b): d = m0 + wm * 128 + 16 a + 4 lq + r
        // of output row n0 + wn * 128 + 16 b + lrow.
        const int64_t m = static_cast<int64_t>(place.m) * kTile + wm * kWaveSide;
        const int m_left = static_cast<int>(p.m - m);  // a multiple of 64, or <= 0
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) {
            const int64_t n =
                static_cast<int64_t>(place.n) * kTile + wn * kWaveSide + 16 * b + lrow;
            if constexpr (kSlab) {
                float* row = p.slabs + (place.split * p.n + n) * p.m + m + 4 * lq;
#pragma unroll
                for (int a = 0; a < kBlocks; ++a) {
                    if (16 * a >= m_left || n >= p.n) continue;
                    const f32x4 x = {value(acc[a][b][0]), value(acc[a][b][1]),
                                     value(acc[a][b][2]), value(acc[a][b][3])};
                    *reinterpret_cast<f32x4*>(row + 16 * a) = x;
                    pin();
                }
            } else {
                // Lane quarters trade halves of two blocks so that each has 8
                // consecutive d: 16 bytes a lane, 64 a row and store.  A
                // row's two stores fill a 128-byte line in L2; as nontemporal
                // stores the training passes at [152064, 3584] were slower
                // (linear step 2832 against 2782 us, head 3761 against 3736).
                uint16_t* row = p.out + n * p.ld_out + m + 8 * lq;
#pragma unroll
                for (int a = 0; a < kBlocks; a += 2) {
                    uint32_t x[2], y[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        x[h] = pack2<DT>(value(acc[a][b][2 * h]), value(acc[a][b][2 * h + 1]));
                        y[h] = pack2<DT>(value(acc[a + 1][b][2 * h]),
                                         value(acc[a + 1][b][2 * h + 1]));
                    }
                    const u32x4 w = gather8(x, y);
                    if (16 * a < m_left && n < p.n)
                        *reinterpret_cast<u32x4*>(row + 16 * a) = w;
                    pin();
                }
            }
        }
    }
    // The last copies (of length 0) write zeros to LDS: before the workgroup
    // gives it up.
    __builtin_amdgcn_s_waitcnt(waitcnt(0, 15));
}

// out = (accumulate ? acc : 0) + the slabs, in slab order; float32 into `acc`,
// or rounded once to 16 bits into `out`.
template <int DT>
__global__ __launch_bounds__(256) void klp_head_sum_kernel(HeadSumParams p) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < p.n_vec;
         i += stride) {
        f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
        if (p.accumulate) s = reinterpret_cast<const f32x4*>(p.acc)[i];
        for (int k = 0; k < p.n_slabs; ++k)
            s += reinterpret_cast<const f32x4*>(p.slabs)[k * p.n_vec + i];
        if (p.out) {
            uint2 w;
            w.x = pack2<DT>(s[0], s[1]);
            w.y = pack2<DT>(s[2], s[3]);
            reinterpret_cast<uint2*>(p.out)[i] = w;
        } else {
            reinterpret_cast<f32x4*>(p.acc)[i] = s;
        }
    }
}

template <int DT>
static hipError_t launch_head_gemm_dt(const HeadGemmParams& p, unsigned grid, hipStream_t stream) {
    if (p.slabs != nullptr)
        return launch_kernel(klp_head_gemm_kernel<DT, false, true>, dim3(grid), dim3(kThreads),
                             stream, p);
    return launch_kernel(klp_head_gemm_kernel<DT, true, false>, dim3(grid), dim3(kThreads), stream,
                         p);
}

hipError_t launch_head_gemm(int dtype, const HeadGemmParams& p, hipStream_t stream) {
    const int64_t items8 = (p.n_items + 7) / 8 * 8;
    const unsigned grid = static_cast<unsigned>(items8 < kHeadGemmCus ? items8 : kHeadGemmCus);
    if (dtype == kBF16) return launch_head_gemm_dt<kBF16>(p, grid, stream);
    if (dtype == kFP16) return launch_head_gemm_dt<kFP16>(p, grid, stream);
    return hipErrorInvalidValue;
}

hipError_t launch_head_sum(int dtype, const HeadSumParams& p, hipStream_t stream) {
    int64_t blocks = (p.n_vec + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    const dim3 grid(static_cast<unsigned>(blocks));
    if (dtype == kBF16) return launch_kernel(klp_head_sum_kernel<kBF16>, grid, dim3(256), stream, p);
    if (dtype == kFP16) return launch_kernel(klp_head_sum_kernel<kFP16>, grid, dim3(256), stream, p);
    return hipErrorInvalidValue;
}

}  // namespace klp
