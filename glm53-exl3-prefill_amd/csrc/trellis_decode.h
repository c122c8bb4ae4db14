// Trellis tile decode for gfx950.
//
// A 16x16 tile is 256 positions; position p's 16-bit state is the window of stream bits
// [(p+1)K - 16, (p+1)K) (mod 256K) of the tile's little-endian dword stream, its first bit as bit 0.
// decode(state): x = state * 0xCBAC1FED mod 2^32; y = (x & 0x8FFF8FFF) ^ 0x3B603B60;
//                w = fp16(y.lo16) + fp16(y.hi16)  (one fp16 add).
// A lane decodes one chunk: the 8 positions p = 8c + j (c = chunk 0..31, j = 0..7), which sit at tile rows
// k = 2(c & 3) + (j & 1) + 8((j >> 1) & 1) and columns n = (c >> 2) + 8(j >> 2).
//
// gfx950 cost per weight. Measured per wave64 instruction and SIMD at four waves per SIMD (2.1-2.4 GHz): v_mul_lo_u32,
// v_mad_u32_u16, v_bfe_u32, v_alignbit_b32 and every SDWA form 2.4 cycles; right shifts, v_and_b32 and v_bitop3_b32
// 1.6-1.7. A full 32-bit product thus costs no more than either half of a product built from 16-bit multiplies, so a
// state is cut out of its dwords by one v_bfe_u32 (a right shift where it is the upper half) and multiplied by one
// v_mul_lo_u32; v_bitop3 does mask-and-xor in one op, and SDWA fp16 adds write each sum into its half of the packed
// output pair in place. About 4.1 VALU ops per weight. A register-only loop of this decode and two MFMAs per 16 weights
// runs 12.3 T weights/s on the device at four waves per SIMD (2.28 GHz), against 10.7 (2.20 GHz) with the product as
// an SDWA 16-bit multiply into the upper word and a v_mad_u32_u16.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace exl3 {

constexpr uint32_t MCG_MUL = 0xCBAC1FEDu;
constexpr uint32_t MCG_XOR = 0x3B603B60u;
constexpr uint32_t MCG_MASK = 0x8FFF8FFFu;

// gfx950 forwards a VALU result written through an SDWA destination select (a partial-register write) to the
// next instruction stale: the consumer must be at least one instruction later. The compiler's hazard recognizer
// cannot see inside an asm statement, so every SDWA result below is consumed only by a VALU instruction of the same
// asm block at least one instruction later, and a block whose last writes are SDWA ends with an s_nop, so whatever the
// compiler places after the block reads them at least one wait state later. Inputs of these blocks must likewise not come
// from instructions with wait-state rules of their own (per-lane 64-bit shifts fed into them gave wrong results at
// random): callers hand them 32-bit funnel shifts, loads and DPP moves.

// The code's two fp16 halves of a state isolated in the low 16 bits.
__device__ __forceinline__ uint32_t mcg_halves(uint32_t state) { return ((state * MCG_MUL) & MCG_MASK) ^ MCG_XOR; }

// Four packed fp16 pairs from eight codes' halves: w[i] = {fp16(y[2i].lo + y[2i].hi), fp16(y[2i+1].lo + y[2i+1].hi)}.
// The low halves are written first (upper half zeroed), then the high halves with the low ones preserved -- each
// read-modify-write four instructions after the write it reads -- and an s_nop guards the last partial write.
__device__ __forceinline__ void add_halves_4pairs(const uint32_t (&y)[8], uint32_t (&w)[4])
{
    asm("v_add_f16_sdwa %0, %4, %4 dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_1\n\t"
        "v_add_f16_sdwa %1, %6, %6 dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_1\n\t"
        "v_add_f16_sdwa %2, %8, %8 dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_1\n\t"
        "v_add_f16_sdwa %3, %10, %10 dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:WORD_0 src1_sel:WORD_1\n\t"
        "v_add_f16_sdwa %0, %5, %5 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0 src1_sel:WORD_1\n\t"
        "v_add_f16_sdwa %1, %7, %7 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0 src1_sel:WORD_1\n\t"
        "v_add_f16_sdwa %2, %9, %9 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0 src1_sel:WORD_1\n\t"
        "v_add_f16_sdwa %3, %11, %11 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:WORD_0 src1_sel:WORD_1\n\t"
        "s_nop 1"
        : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3])
        : "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]), "v"(y[4]), "v"(y[5]), "v"(y[6]), "v"(y[7]));
}

// Decoded chunk, as four packed fp16 pairs ordered for a [n][k] (k-contiguous) destination:
//   out[0] = (k0, k0+1) at column n0, out[1] = (k0+8, k0+9) at n0, out[2] = (k0, k0+1) at n0+8,
//   out[3] = (k0+8, k0+9) at n0+8, with k0 = 2(c & 3), n0 = c >> 2.
struct Chunk4 { uint32_t w[4]; };

// The 16-bit state starting OFF bits into hi:lo, from lo, hi or the dword across them (mid = bits 16 .. 47).
template <int OFF>
__device__ __forceinline__ uint32_t state_at(uint32_t lo, uint32_t mid, uint32_t hi)
{
    static_assert(OFF >= 0 && OFF <= 48, "a state within 64 bits");
    if constexpr (OFF <= 16) return (lo >> OFF) & 0xFFFF;
    else if constexpr (OFF <= 32) return (mid >> (OFF - 16)) & 0xFFFF;
    else return (hi >> (OFF - 32)) & 0xFFFF;
}

// Decode the chunk whose stream bits sit in hi:lo starting at bit OFF (BITS in {1,2,3,4}).
template <int BITS, int OFF>
__device__ __forceinline__ Chunk4 decode_chunk(uint32_t lo, uint32_t hi)
{
    const uint32_t mid = __builtin_amdgcn_alignbit(hi, lo, 16);
    const uint32_t y[8] = {mcg_halves(state_at<OFF>(lo, mid, hi)), mcg_halves(state_at<OFF + BITS>(lo, mid, hi)),
                           mcg_halves(state_at<OFF + 2 * BITS>(lo, mid, hi)),
                           mcg_halves(state_at<OFF + 3 * BITS>(lo, mid, hi)),
                           mcg_halves(state_at<OFF + 4 * BITS>(lo, mid, hi)),
                           mcg_halves(state_at<OFF + 5 * BITS>(lo, mid, hi)),
                           mcg_halves(state_at<OFF + 6 * BITS>(lo, mid, hi)),
                           mcg_halves(state_at<OFF + 7 * BITS>(lo, mid, hi))};
    Chunk4 c;
    add_halves_4pairs(y, c.w);
    return c;
}

// Decode four dwords of two independent states each -> packed fp16 pairs, one dword per input dword.
__device__ __forceinline__ void decode_states_4(const uint32_t (&r)[4], uint32_t (&w)[4])
{
    uint32_t y[8];
    #pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        y[2 * i] = mcg_halves(r[i] & 0xFFFF);
        y[2 * i + 1] = mcg_halves(r[i] >> 16);
    }
    add_halves_4pairs(y, w);
}

}  // namespace exl3
