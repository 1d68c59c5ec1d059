// klp_mfma.h — matrix-core building blocks shared by the LM head kernels
// (klp_lmhead.hip, klp_head_gemm.hip): 256 x 256 output tiles on four waves,
// each 128 x 128 of them as 8 x 8 blocks of v_mfma_f32_16x16x32, fed through
// LDS rings of 64-column (K) stages.
#pragma once

#include "klp_device.h"

namespace klp {
namespace mfma {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
// One operand register block: 8 consecutive K values of one row, 16 bits each.
typedef u32x4 operand;

constexpr int kThreads = 256;
constexpr int kBlocks = 8;               // 16-wide blocks per wave and side
constexpr int kWaveSide = kBlocks * 16;  // 128
constexpr int kTile = 2 * kWaveSide;     // 256: two waves along each side
constexpr int kBK = 64;                  // K per stage
constexpr int kRowBytes = kBK * 2;
constexpr int kSlotBytes = kTile * kRowBytes;
// All 160 KB of LDS: a ring of 3 stages of one operand, 2 of the other.
constexpr int kASlots = 3;
constexpr int kBSlots = 2;
constexpr int kLdsBytes = (kASlots + kBSlots) * kSlotBytes;
static_assert(kLdsBytes <= 160 * 1024, "LDS holds 160 KB");
// One copy moves 64 lanes x 16 B = 1 KB; 8 per wave fill a slot.
constexpr int kCopies = 8;

typedef __attribute__((address_space(3))) void lds_void;

// s_waitcnt immediate: vmcnt <= vm, lgkmcnt <= lgkm (15: no wait).
constexpr int waitcnt(int vm, int lgkm) {
    return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | (lgkm << 8);
}

// Keeps what is written before it before what is written after it.
__device__ __forceinline__ void pin() { __builtin_amdgcn_sched_barrier(0); }

// acc += a * b (`zero`: acc = a * b), in AGPRs and in place: left to the
// builtin, the compiler renames the 256 accumulators from MFMA to MFMA and
// pays for it in moves through VGPRs and spills at every join (436-920 bytes
// of scratch in the LM head's forward, 970 against 800 us).  The wait states
// it would insert around its own MFMAs are then the caller's: the operands
// come straight from LDS reads (waited for as any use), so that no VALU
// instruction writes one in the 2 wait states before; an accumulator's own
// MFMAs are a half stage apart, 64 or, with blocks of 192 or 128 tokens, 48
// or 32; and
// drain() comes before other instructions read accumulators.  The compiler
// is free to move a register in between: tests/test_mfma_hazards_cpu.py looks
// for that in the generated code.
template <int DT>
__device__ __forceinline__ void mul_add(f32x4& acc, operand a, operand b, bool zero) {
    if constexpr (DT == kBF16) {
        if (zero)  // a constant at every call
            asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc) : "v"(a), "v"(b));
        else
            asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
    } else {
        if (zero)
            asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(acc) : "v"(a), "v"(b));
        else
            asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
    }
}

// An accumulator's value, read where it is needed (the compiler would move
// more than half of them to VGPRs ahead of an epilogue, and spill).
__device__ __forceinline__ float value(float acc) {
    float v;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(acc));
    return v;
}

// The wait states between the last MFMA and a VALU read of its result (11 for
// an MFMA of 8 passes; these are busy for 16 cycles, 4 passes), rounded up.
__device__ __forceinline__ void drain() { asm volatile("s_nop 15\n\ts_nop 7"); }

// Two floats rounded to DT and packed, the first in the low half.
template <int DT> __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    if constexpr (DT == kBF16)
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
    else
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, f16x2));
}

// Two floats rounded to DT's values.
template <int DT> __device__ __forceinline__ void round2(float& a, float& b) {
    const uint32_t w = pack2<DT>(a, b);
    a = to_f32<DT>(static_cast<uint16_t>(w));
    b = to_f32<DT>(static_cast<uint16_t>(w >> 16));
}

// Lane quarter q holds 4 consecutive 16-bit values of block a (`x`, two to a
// word) and of block a + 1 (`y`), at 4 q of each block's 16.  Returns 8
// consecutive ones: quarters 0 and 1 get block a's first and second half, 2
// and 3 block a + 1's (8 q of the two blocks' 32).
__device__ __forceinline__ u32x4 gather8(const uint32_t (&x)[2], const uint32_t (&y)[2]) {
    u32x4 r;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const auto s = __builtin_amdgcn_permlane32_swap(x[h], y[h], false, false);
        const auto t = __builtin_amdgcn_permlane16_swap(s[0], s[1], false, false);
        r[h] = t[0];
        r[2 + h] = t[1];
    }
    return r;
}

// K-contiguous operand rows in LDS: slot row r is 128 bytes, its 16-byte
// chunk c at chunk c ^ swz(r).  An operand read (ds_read_b128: row l % 16,
// chunk l / 16 of a half stage in lane l) is served 16 lanes at a time, lanes
// 0-3, 12-15, 20-27 first: rows 0-3 and 12-15 of one chunk with rows 4-11 of
// the next.  Rows of one parity share a 128-byte half of the banks; with
// r / 2 their 8 places differ in every such group, and in groups of
// consecutive lanes.  ((r & 7) ^ (r / 8 & 1) conflicted 2 ways: half of the
// reads' LDS cycles, by SQ_LDS_BANK_CONFLICT.)
__device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }

// K-strided operand rows in LDS: slot row k (of 64) is 512 bytes, 256
// columns; within each 256-byte half its 32-byte block i (16 columns) sits at
// block i ^ swz_k(k).  A transposing read (ds_read_b64_tr_b16) takes, per 16
// lanes, one block of 4 consecutive k; 32 lanes meet k, k + 1, k + 2, k + 3
// and the same + 8: 8 blocks at 8 places, every bank once.
__device__ __forceinline__ int swz_k(int k) { return (k & 3) | (((k >> 3) & 1) << 2); }

// One wave's 1 KB copy to LDS byte offset `lds`: lane l's 16 bytes at `rsrc`
// + voff + soff go to lds + 16 l; past the descriptor's end they are zeros.
// In asm because the compiler, which cannot tell the rings' slots apart, puts
// s_waitcnt vmcnt(0) between a copy it knows of and a following transposing
// read; nothing is loaded into registers here, and the callers count their
// copies and wait for them (also before the kernel ends).  The compiler sees
// no memory instruction, so its wait states are ours: the s_nop is the 1 from
// writing M0 to a copy that reads it; of the 5 from a VALU instruction that
// wrote the descriptor or an offset (the reload of a spilled SGPR) it is the
// second.  All 5 here (s_nop 3) cost the training passes at [152064, 3584]
// 1.3% (head 3727 -> 3778 us, linear step 2768 -> 2805).  In the generated
// code no such write stands that close, and M0, which cannot be named as
// clobbered (it is reserved), has no other use in the kernel that calls this:
// tests/test_mfma_hazards_cpu.py checks both.
__device__ __forceinline__ void copy_to_lds(u32x4 rsrc, uint32_t lds, uint32_t voff, uint32_t soff) {
    asm volatile(
        "s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
        :
        : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff)
        : "memory");
}
// Descriptor of `bytes` bytes at `base` (word 3: dword data).
__device__ __forceinline__ u32x4 bytes_rsrc(const void* base, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    return u32x4{static_cast<uint32_t>(a), static_cast<uint32_t>(a >> 32) & 0xFFFFu, bytes,
                 0x00020000u};
}

// Transposing read: of each 16 lanes, lane j addresses 4 columns
// 4 (j % 4) .. + 3 of row k + j / 4; lane i receives column i of rows k .. k + 3.
__device__ __forceinline__ s16x4 read_tr(const unsigned char* lds) {
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)lds);
}

}  // namespace mfma
}  // namespace klp
