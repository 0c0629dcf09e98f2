// gemm_split.h — the tile of the grouped expert GEMMs: fp32 operands as sums
// of three bfloat16 terms, multiplied on the bf16 matrix cores of gfx950.
//
// x = h + m + l with h = bf16(x), m = bf16(x - h), l = bf16(x - h - m), each
// rounded to nearest: 8 + 8 + 8 significant bits hold all 24 of a float, and
// both subtractions are exact, so for 2^-109 <= |x| < 2^128 - 2^119 (and 0)
// the split loses nothing.  A product takes
// the six terms down to 2^-16 of the largest (hh, hm, mh, mm, hl, lh); the
// three left out are below 2^-25 of it, under half an ulp of the float
// product.  All six go into one float accumulator.  Six
// v_mfma_f32_32x32x16_bf16 (192 cycles) replace eight v_mfma_f32_32x32x2f32
// (512 cycles).  Relative error (2-norm) of 32 x 32 products of N(0, 1) by
// N(0, 0.02) against float64, this against the fp32 MFMA chain: K = 64
// 1.0e-7 / 1.4e-7, 512 3.4e-7 / 4.0e-7, 2048 7.0e-7 / 7.8e-7, 8192 1.4e-6 /
// 1.6e-6 (fewer roundings of the running sum: 6 for 16 products, not 16).
// With only a few nonzero products the terms left out show: four of 64
// 6.3e-8 / 3.8e-8.
//
// Work: 128 x BN tiles (BN = 64 WN) on four waves, WM x WN of (128 / WM) x
// 64; two such workgroups share a CU, so one's splitting and LDS traffic run
// under the other's MFMAs.  Per step of 16 k:
//   B  goes from memory straight to the wave that owns its 64 columns (the
//      packed 1 KB units are four 256-byte runs per load) and is split there;
//      with WM = 1 no other wave needs it;
//   A  (128 rows, gathered) is split once by the workgroup, each thread 4 k
//      of 2 rows, and kept in LDS as three planes in MFMA operand order (two
//      stages of 12 KB, one barrier per step).
// The operands of the next step (128- and 64-column tiles: of the next two) are
// in flight while a step multiplies.
//
// Outside that range the split is not used for the result.  An infinity or
// NaN among the operands makes NaNs of the remainders where the float sum may
// be an infinity, and a float above the largest bfloat16 becomes one; under
// 2^-109 the third term, then the second, falls below bfloat16's smallest
// subnormal (2^-133).  So a sum that is not finite, or nonzero and below
// 2^-80, is computed again on the fp32 MFMAs.  The choice is made element by
// element: no other row's or column's values change an element's bits.  What
// stays less exact than float products: an operand below 2^-109 that meets one
// above 2^29 (its sum may pass 2^-80), and one below 2^-134, which counts as
// zero where a whole sum has no larger ones.  (A layer whose gate sums and H
// are of the order of 2^-118, d = 256, F = 512: 5.6e-5 from float64 without
// the rule, below 3e-6 with it.)
#pragma once
#include "moe_internal.h"
#include "moe_math.h"
#include <type_traits>

namespace moe {
namespace split {

typedef float fx4 __attribute__((ext_vector_type(4)));
typedef float fx16 __attribute__((ext_vector_type(16)));
typedef float fx2 __attribute__((ext_vector_type(2)));
typedef unsigned ux4 __attribute__((ext_vector_type(4)));
typedef unsigned ux2 __attribute__((ext_vector_type(2)));
typedef __bf16 bx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bx8 __attribute__((ext_vector_type(8)));

// Two floats as three packed bf16 pairs.
__device__ __forceinline__ void split2(float x0, float x1, unsigned &h, unsigned &m, unsigned &l) {
    h = __builtin_bit_cast(unsigned, __builtin_convertvector((fx2){x0, x1}, bx2));
    const float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xffff0000u);
    m = __builtin_bit_cast(unsigned, __builtin_convertvector((fx2){r0, r1}, bx2));
    const float q0 = r0 - __uint_as_float(m << 16), q1 = r1 - __uint_as_float(m & 0xffff0000u);
    l = __builtin_bit_cast(unsigned, __builtin_convertvector((fx2){q0, q1}, bx2));
}

// Eight consecutive k of one row or column as the three terms' operands.
struct Frag {
    ux4 t[3];
};
__device__ __forceinline__ Frag split8(fx4 a, fx4 b) {
    Frag f;
    unsigned h, m, l;
#define MOE_SPLIT_PAIR(q, x0, x1)                \
    split2(x0, x1, h, m, l);                     \
    f.t[0][q] = h; f.t[1][q] = m; f.t[2][q] = l;
    MOE_SPLIT_PAIR(0, a[0], a[1])
    MOE_SPLIT_PAIR(1, a[2], a[3])
    MOE_SPLIT_PAIR(2, b[0], b[1])
    MOE_SPLIT_PAIR(3, b[2], b[3])
#undef MOE_SPLIT_PAIR
    return f;
}

__device__ __forceinline__ fx16 mma(ux4 a, ux4 b, fx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bx8, a),
                                                   __builtin_bit_cast(bx8, b), c, 0, 0, 0);
}

// A sum of split products to be replaced by the sum of float products.
constexpr float kSmallSum = 0x1p-80f;
__device__ __forceinline__ bool float_sum_needed(float s) {
    return !(fabsf(s) >= kSmallSum && fabsf(s) <= 0x1.fffffep127f) && s != 0.0f;
}

// Whether a wave has such sums: chk stays 0 while they are finite, lo is the
// smallest 2 |bits| - 1, the largest number for a zero (five VALU instructions
// for two sums; asking each sum the question above cost the backward of T =
// 1000, d = 1024, F = 512, E = 64, top-4 10 us of 770).
struct SumCheck {
    float chk = 0.0f;
    unsigned lo = ~0u;
    __device__ __forceinline__ void add(fx16 a) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            chk = fmaf(a[r], 0.0f, chk);
            lo = min(lo, (__float_as_uint(a[r]) << 1) - 1u);
        }
    }
    __device__ __forceinline__ bool fits() const {
        return !__ballot(!(chk == 0.0f) || lo < (__float_as_uint(kSmallSum) << 1) - 1u);
    }
};

// The six term pairs, smallest first.
constexpr int kPairs = 6;
__device__ constexpr int kPairA[kPairs] = {2, 0, 1, 1, 0, 0};
__device__ constexpr int kPairB[kPairs] = {0, 2, 1, 0, 1, 0};

constexpr int kStageBytes = 3 * 128 * 32;        // three planes of 128 rows x 16 k
constexpr int kTileLds = 2 * kStageBytes;

}  // namespace split
}  // namespace moe
