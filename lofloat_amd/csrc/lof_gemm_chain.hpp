// lof_gemm_chain.hpp -- emulated-accumulation GEMM tile for chunks of 1 to 32 (gfx950): chunk
// sums of 2 to 32 products on the f32 matrix cores, chunk 1 leaf by leaf.
//
// For chunk c > 1 the rule is: p = FP32 fmaf chain over the chunk's c products in ascending
// k, from +0, then acc <- round(RTO24(p + acc)).  v_mfma_f32_32x32x2_f32 and
// v_mfma_f32_16x16x4_f32 are that chain: each of their k steps is one fused multiply-add,
// rounded to nearest even, FP32 subnormals kept, in ascending k, whatever the wave's rounding
// mode.  Measured on gfx950, bit for bit against the fmaf chain: no difference in 4.4e9
// outputs of 4 to 32 k, from +0 and from random accumulators, over uniform, 60-binade and
// all-exponent operands, FP32-subnormal operands and products, near-cancelling sums, small
// integers with zeros, overflowing products, infinities and NaN (NaN as a class)
// (test_gemm_chain_gpu.py repeats such a comparison).  So a chunk sum needs no exactness proof,
// no operand statistics and no VALU multiply-adds: the matrix cores run it at twice the VALU's
// FP32 rate (153 TFLOP/s measured) and leave the VALU to the leaves.
//
// The leaf takes any finite p and acc with no test:
//   mantissa-only, 1..22 bits   the two directed roundings of p + acc, of which the odd one is
//                               RTO24's result (rto_fma16), then round-to-nearest-even at a fixed
//                               bit of the pattern: 7 instructions;
//   mantissa-only, 23 bits      the odd one is the result: 4 instructions;
//   binary16-shaped             one mixed-precision FMA, which rounds the exact -acc - p once to
//                               binary16, and one conversion; results that reach the format's
//                               top binade (or 2^15) redo the leaf in its general form.
// A slice with an infinity or a NaN among its operands has the NaN sums brought to one pattern
// before the leaf, so that rounding cannot carry a payload out of the NaN range.
//
// Chunk 1 (acc <- round(RTO24(a b + acc)) for every k) works on the negated accumulators; what
// bounds it is VALU issue.  Cycles a wave on gfx950, measured with four waves a SIMD: FP32 add,
// multiply, FMA and 32-bit logic 2.5 to 3, v_bfi_b32, v_bfe_i32, conversions and v_pk_fma_f16
// (two leaves) 4.4, v_fma_mixlo_f16 and v_min3_f16 8.4, v_min_f16 2.6.  By accumulator:
//   any mantissa                two directed FMAs and the odd one of them (rto_fnma16), 15 cycles a
//                               leaf, and three instructions more below 23 bits;
//   23 bits, exact sums         the f32 MFMA (4 cycles a leaf);
//   binary16-shaped, 10 bits    one binary16 FMA on binary16 operands, two leaves an instruction,
//                               from slices kept as binary16 pairs (2.2 cycles a leaf); one
//                               mixed FMA on FP32 operands (8.4; 10 bits: 2.6 more for the check).
// e4m3 operands, before and after the slices were kept as binary16 pairs, 10 bits: 4096^3 3.68 ->
// 2.28 ms, 1000x768x3072 293 -> 196 us, 128x25088x1152 301 -> 190 us; binary16-shaped: 2.86 -> 1.84
// ms, 216 -> 133 us, 243 -> 152 us.
//
// Tile: 4 waves, each WMB x WNB blocks of BS x BS outputs (BS = 32, or 16 for products with few
// outputs, where a 32-row block would leave most of the chip idle).  A and B slices of BK k sit
// k-major in double-buffered LDS; the next slice loads into registers while the current one
// computes.  Rows past the matrix repeat its last row; k past K is (-0) * (+0) = -0, which adds
// nothing to a chain, signs of zero included.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "lof_gemm_mfma.hpp"

namespace lofamd {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Accumulators the tile's leaf takes (ChainArgs-free: the constants are GemmArgs').
enum ChainKind : int { kChainMant = 0, kChainMant23 = 1, kChainHalf = 2, kChainMant10 = 3 };

// An operand slice in LDS: R rows (A's m, B's n) by BK k, k-major in groups of four k that
// start PAD floats apart, the row swizzled by k.  An MFMA operand read takes KI consecutive k of
// 64 / KI consecutive rows each; the swizzle puts them in different banks (64 banks of 4
// bytes), and PAD spreads the transposing stores of a row-major operand, whose lanes hold
// consecutive groups of four k, to two-way conflicts.  (Rows of R + 4 floats: every operand read had
// them.  4096^3, chunk 32, both operands row-major: 67 M conflict cycles of 268 M LDS ones, two a store.)
template <int R, int BK, int KI>
struct ChainLds {
    static constexpr int PAD = R >= 64 && KI == 2 ? 8 : 4;
    static constexpr int GROUP = 4 * R + PAD;
    static constexpr int FLOATS = BK / 4 * GROUP;
    static __device__ __forceinline__ constexpr int swz(int k) {   // multiples of 16
        return KI == 2 ? 32 * (k & 1) : R >= 64 ? 16 * (k & 3) : R == 32 ? 16 * ((k >> 1) & 1) : 0;
    }
    static __device__ __forceinline__ constexpr int row(int k) { return (k >> 2) * GROUP + (k & 3) * R; }
};

template <int BS_, int WR_, int WC_, int WMB_, int WNB_, int BK_>
struct ChainTile {
    static constexpr int BS = BS_, WR = WR_, WC = WC_, WMB = WMB_, WNB = WNB_, BK = BK_;
    static_assert(WR * WC == 4 && (BS == 16 || BS == 32), "four waves of MFMA blocks");
    static constexpr int BM = WR * WMB * BS, BN = WC * WNB * BS;
    static constexpr int NR = BS * BS / 64;        // outputs per lane and block
    static constexpr int KI = BS == 32 ? 2 : 4;    // k per MFMA
    static constexpr int BUF_FLOATS = ChainLds<BM, BK, KI>::FLOATS + ChainLds<BN, BK, KI>::FLOATS;
    static constexpr int SMEM_FLOATS = 2 * BUF_FLOATS + 44;   // + 3 flags, statistics, 2 x 3 flags
    static constexpr int NA4 = BM * BK / 1024, NB4 = BN * BK / 1024;   // float4 per thread
    static_assert(NA4 * 1024 == BM * BK && NB4 * 1024 == BN * BK, "whole float4s per thread");
};

// Four consecutive floats from a pointer with a float's alignment: global memory takes
// dword-aligned 16-byte loads, so odd leading dimensions and sub-views need no scalar path.
__device__ __forceinline__ float4 gld4u(const float* p) {
    typedef float v4 __attribute__((ext_vector_type(4), aligned(4)));
    const v4 v = *(const __attribute__((address_space(1))) v4*)p;
    return make_float4(v.x, v.y, v.z, v.w);
}

// acc[o] <- RTO24(acc[o] + p[o]) as rto_fma16, for 4 and 8 outputs
__device__ __forceinline__ void rto_add4(const float* p, float* acc) {
    float rd[4], mask[4];
    asm volatile(
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 2\n\t"
        "s_nop 1\n\t"
        "v_add_f32 %4, %0, %12\n\t"
        "v_add_f32 %5, %1, %13\n\t"
        "v_add_f32 %6, %2, %14\n\t"
        "v_add_f32 %7, %3, %15\n\t"
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 1\n\t"
        "s_nop 1\n\t"
        "v_add_f32 %0, %0, %12\n\t"
        "v_add_f32 %1, %1, %13\n\t"
        "v_add_f32 %2, %2, %14\n\t"
        "v_add_f32 %3, %3, %15\n\t"
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0\n\t"
        "v_bfe_i32 %8, %0, 0, 1\n\t"
        "v_bfe_i32 %9, %1, 0, 1\n\t"
        "v_bfe_i32 %10, %2, 0, 1\n\t"
        "v_bfe_i32 %11, %3, 0, 1\n\t"
        "v_bfi_b32 %0, %8, %0, %4\n\t"
        "v_bfi_b32 %1, %9, %1, %5\n\t"
        "v_bfi_b32 %2, %10, %2, %6\n\t"
        "v_bfi_b32 %3, %11, %3, %7"
        : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]),
          "=&v"(rd[0]), "=&v"(rd[1]), "=&v"(rd[2]), "=&v"(rd[3]),
          "=&v"(mask[0]), "=&v"(mask[1]), "=&v"(mask[2]), "=&v"(mask[3])
        : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]));
}

__device__ __forceinline__ void rto_add8(const float* p, float* acc) {
    float rd[8], mask[4];
    asm volatile(
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 2\n\t"
        "s_nop 1\n\t"
        "v_add_f32 %8, %0, %20\n\t"
        "v_add_f32 %9, %1, %21\n\t"
        "v_add_f32 %10, %2, %22\n\t"
        "v_add_f32 %11, %3, %23\n\t"
        "v_add_f32 %12, %4, %24\n\t"
        "v_add_f32 %13, %5, %25\n\t"
        "v_add_f32 %14, %6, %26\n\t"
        "v_add_f32 %15, %7, %27\n\t"
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 1\n\t"
        "s_nop 1\n\t"
        "v_add_f32 %0, %0, %20\n\t"
        "v_add_f32 %1, %1, %21\n\t"
        "v_add_f32 %2, %2, %22\n\t"
        "v_add_f32 %3, %3, %23\n\t"
        "v_add_f32 %4, %4, %24\n\t"
        "v_add_f32 %5, %5, %25\n\t"
        "v_add_f32 %6, %6, %26\n\t"
        "v_add_f32 %7, %7, %27\n\t"
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0\n\t"
        "v_bfe_i32 %16, %0, 0, 1\n\t"
        "v_bfe_i32 %17, %1, 0, 1\n\t"
        "v_bfe_i32 %18, %2, 0, 1\n\t"
        "v_bfe_i32 %19, %3, 0, 1\n\t"
        "v_bfi_b32 %0, %16, %0, %8\n\t"
        "v_bfi_b32 %1, %17, %1, %9\n\t"
        "v_bfi_b32 %2, %18, %2, %10\n\t"
        "v_bfi_b32 %3, %19, %3, %11\n\t"
        "v_bfe_i32 %16, %4, 0, 1\n\t"
        "v_bfe_i32 %17, %5, 0, 1\n\t"
        "v_bfe_i32 %18, %6, 0, 1\n\t"
        "v_bfe_i32 %19, %7, 0, 1\n\t"
        "v_bfi_b32 %4, %16, %4, %12\n\t"
        "v_bfi_b32 %5, %17, %5, %13\n\t"
        "v_bfi_b32 %6, %18, %6, %14\n\t"
        "v_bfi_b32 %7, %19, %7, %15"
        : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]),
          "+v"(acc[4]), "+v"(acc[5]), "+v"(acc[6]), "+v"(acc[7]),
          "=&v"(rd[0]), "=&v"(rd[1]), "=&v"(rd[2]), "=&v"(rd[3]),
          "=&v"(rd[4]), "=&v"(rd[5]), "=&v"(rd[6]), "=&v"(rd[7]),
          "=&v"(mask[0]), "=&v"(mask[1]), "=&v"(mask[2]), "=&v"(mask[3])
        : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]),
          "v"(p[4]), "v"(p[5]), "v"(p[6]), "v"(p[7]));
}

// binary16(na - p), one rounding of the exact difference (see mix_sub16x16), as a float
__device__ __forceinline__ float mix_sub16(float na, float p) {
    _Float16 r;
    asm("v_fma_mixlo_f16 %0, %1, -1.0, %2 op_sel_hi:[0,0,0]" : "=v"(r) : "v"(p), "v"(na));
    return (float)r;
}

// The leaves below read MFMA results inside asm statements, where the compiler does not insert the
// wait states that a vector read of an MFMA result needs (18 after a 16-pass MFMA): this
// statement waits 20 and hands the results on.
template <class V>
__device__ __forceinline__ void mfma_settle(V& a) {
    asm volatile("s_nop 15\n\ts_nop 3" : "+v"(a));
}
template <class V>
__device__ __forceinline__ void mfma_settle(V& a, V& b) {
    asm volatile("s_nop 15\n\ts_nop 3" : "+v"(a), "+v"(b));
}
template <class V>
__device__ __forceinline__ void mfma_settle(V& a, V& b, V& c, V& d) {
    asm volatile("s_nop 15\n\ts_nop 3" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
}

// The general leaf of a binary16-shaped accumulator on its negated form, out of line: reached
// only by results in the format's top binade or past it.
__device__ __noinline__ float chain_half_slow(float p, float na, LeafGen L) {
    return -leaf_f_slow(p, -na, L);
}

// The leaves of NR (4 or 8) outputs of a chunk.  acc: the accumulators (kChainHalf: negated).
// inside(o), wave-uniform: output o of some lane lies in the matrix.  Outputs past its edges repeat a
// row or a column of it and are dropped: on their own they never take the general leaf
// (sums past the top binade, chunk 2, 64x64 tile, us: 3x40000x256 5572 -> 872, 20x40000x256
// 5611 -> 3105).
template <int KIND, int NR, class Inside>
__device__ __forceinline__ void chain_leaves(float (&p)[NR], float (&acc)[NR], bool special,
                                             const GemmArgs& g, Inside inside) {
    if constexpr (KIND == kChainHalf) {
        float t[NR], top = 0.0f;
#pragma unroll
        for (int o = 0; o < NR; ++o) {
            t[o] = mix_sub16(acc[o], p[o]);
            top = fmaxf(top, fabsf(t[o]));
        }
        if (__builtin_expect(__any(top >= g.half_top), 0)) {
#pragma unroll
            for (int o = 0; o < NR; ++o)
                if (inside(o) && fabsf(t[o]) >= g.half_top)
                    t[o] = chain_half_slow(p[o], acc[o], leaf_gen(g));
        }
#pragma unroll
        for (int o = 0; o < NR; ++o) acc[o] = t[o];
    } else {
        if constexpr (KIND == kChainMant)
            if (special) {   // wave-uniform: a NaN sum to the one quiet pattern
#pragma unroll
                for (int o = 0; o < NR; ++o)
                    p[o] = p[o] != p[o] ? __uint_as_float(0x7FC00000u) : p[o];
            }
        if constexpr (NR == 8) rto_add8(p, acc);
        else rto_add4(p, acc);
        if constexpr (KIND == kChainMant) {
#pragma unroll
            for (int o = 0; o < NR; ++o) {
                const uint32_t t = __float_as_uint(acc[o]);
                acc[o] = __uint_as_float((t + g.dr_half + __builtin_amdgcn_ubfe(t, g.dr_rf, 1u)) &
                                         g.dr_mask);
            }
        }
    }
}

// Chunk 1, on the negated accumulator: na[o] <- -RTO24(a[o] * b + acc[o]), na = -acc.  Round-to-odd
// and both roundings after it are odd functions, so rto_fma16's construction applied to
// y = na - a b gives the negated result; only an exact zero changes: -(RTO24's zero of the sum)
// is roundTowardPositive's zero of y, so the pick is by rd's last bit and falls to ru.
__device__ __forceinline__ void rto_fnma16(const float* a, const float* b, float* na) {
    float rd[16], mask[4];
    asm volatile(
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 2\n\t"
        "s_nop 1\n\t"
        "v_fma_f32 %16, -%36, %52, %0\n\t"
        "v_fma_f32 %17, -%37, %53, %1\n\t"
        "v_fma_f32 %18, -%38, %54, %2\n\t"
        "v_fma_f32 %19, -%39, %55, %3\n\t"
        "v_fma_f32 %20, -%40, %56, %4\n\t"
        "v_fma_f32 %21, -%41, %57, %5\n\t"
        "v_fma_f32 %22, -%42, %58, %6\n\t"
        "v_fma_f32 %23, -%43, %59, %7\n\t"
        "v_fma_f32 %24, -%44, %60, %8\n\t"
        "v_fma_f32 %25, -%45, %61, %9\n\t"
        "v_fma_f32 %26, -%46, %62, %10\n\t"
        "v_fma_f32 %27, -%47, %63, %11\n\t"
        "v_fma_f32 %28, -%48, %64, %12\n\t"
        "v_fma_f32 %29, -%49, %65, %13\n\t"
        "v_fma_f32 %30, -%50, %66, %14\n\t"
        "v_fma_f32 %31, -%51, %67, %15\n\t"
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 1\n\t"
        "s_nop 1\n\t"
        "v_fma_f32 %0, -%36, %52, %0\n\t"
        "v_fma_f32 %1, -%37, %53, %1\n\t"
        "v_fma_f32 %2, -%38, %54, %2\n\t"
        "v_fma_f32 %3, -%39, %55, %3\n\t"
        "v_fma_f32 %4, -%40, %56, %4\n\t"
        "v_fma_f32 %5, -%41, %57, %5\n\t"
        "v_fma_f32 %6, -%42, %58, %6\n\t"
        "v_fma_f32 %7, -%43, %59, %7\n\t"
        "v_fma_f32 %8, -%44, %60, %8\n\t"
        "v_fma_f32 %9, -%45, %61, %9\n\t"
        "v_fma_f32 %10, -%46, %62, %10\n\t"
        "v_fma_f32 %11, -%47, %63, %11\n\t"
        "v_fma_f32 %12, -%48, %64, %12\n\t"
        "v_fma_f32 %13, -%49, %65, %13\n\t"
        "v_fma_f32 %14, -%50, %66, %14\n\t"
        "v_fma_f32 %15, -%51, %67, %15\n\t"
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0\n\t"
        "v_bfe_i32 %32, %16, 0, 1\n\t"
        "v_bfe_i32 %33, %17, 0, 1\n\t"
        "v_bfe_i32 %34, %18, 0, 1\n\t"
        "v_bfe_i32 %35, %19, 0, 1\n\t"
        "v_bfi_b32 %0, %32, %16, %0\n\t"
        "v_bfi_b32 %1, %33, %17, %1\n\t"
        "v_bfi_b32 %2, %34, %18, %2\n\t"
        "v_bfi_b32 %3, %35, %19, %3\n\t"
        "v_bfe_i32 %32, %20, 0, 1\n\t"
        "v_bfe_i32 %33, %21, 0, 1\n\t"
        "v_bfe_i32 %34, %22, 0, 1\n\t"
        "v_bfe_i32 %35, %23, 0, 1\n\t"
        "v_bfi_b32 %4, %32, %20, %4\n\t"
        "v_bfi_b32 %5, %33, %21, %5\n\t"
        "v_bfi_b32 %6, %34, %22, %6\n\t"
        "v_bfi_b32 %7, %35, %23, %7\n\t"
        "v_bfe_i32 %32, %24, 0, 1\n\t"
        "v_bfe_i32 %33, %25, 0, 1\n\t"
        "v_bfe_i32 %34, %26, 0, 1\n\t"
        "v_bfe_i32 %35, %27, 0, 1\n\t"
        "v_bfi_b32 %8, %32, %24, %8\n\t"
        "v_bfi_b32 %9, %33, %25, %9\n\t"
        "v_bfi_b32 %10, %34, %26, %10\n\t"
        "v_bfi_b32 %11, %35, %27, %11\n\t"
        "v_bfe_i32 %32, %28, 0, 1\n\t"
        "v_bfe_i32 %33, %29, 0, 1\n\t"
        "v_bfe_i32 %34, %30, 0, 1\n\t"
        "v_bfe_i32 %35, %31, 0, 1\n\t"
        "v_bfi_b32 %12, %32, %28, %12\n\t"
        "v_bfi_b32 %13, %33, %29, %13\n\t"
        "v_bfi_b32 %14, %34, %30, %14\n\t"
        "v_bfi_b32 %15, %35, %31, %15\n\t"
        "s_nop 1"
        : "+v"(na[0]), "+v"(na[1]), "+v"(na[2]), "+v"(na[3]),
          "+v"(na[4]), "+v"(na[5]), "+v"(na[6]), "+v"(na[7]),
          "+v"(na[8]), "+v"(na[9]), "+v"(na[10]), "+v"(na[11]),
          "+v"(na[12]), "+v"(na[13]), "+v"(na[14]), "+v"(na[15]),
          "=&v"(rd[0]), "=&v"(rd[1]), "=&v"(rd[2]), "=&v"(rd[3]),
          "=&v"(rd[4]), "=&v"(rd[5]), "=&v"(rd[6]), "=&v"(rd[7]),
          "=&v"(rd[8]), "=&v"(rd[9]), "=&v"(rd[10]), "=&v"(rd[11]),
          "=&v"(rd[12]), "=&v"(rd[13]), "=&v"(rd[14]), "=&v"(rd[15]),
          "=&v"(mask[0]), "=&v"(mask[1]), "=&v"(mask[2]), "=&v"(mask[3])
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]),
          "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]),
          "v"(a[8]), "v"(a[9]), "v"(a[10]), "v"(a[11]),
          "v"(a[12]), "v"(a[13]), "v"(a[14]), "v"(a[15]),
          "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]),
          "v"(b[4]), "v"(b[5]), "v"(b[6]), "v"(b[7]),
          "v"(b[8]), "v"(b[9]), "v"(b[10]), "v"(b[11]),
          "v"(b[12]), "v"(b[13]), "v"(b[14]), "v"(b[15]));
}

__device__ __forceinline__ void rto_fnma4(const float* a, const float* b, float* na) {
    float rd[4], mask[4];
    asm volatile(
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 2\n\t"
        "s_nop 1\n\t"
        "v_fma_f32 %4, -%12, %16, %0\n\t"
        "v_fma_f32 %5, -%13, %17, %1\n\t"
        "v_fma_f32 %6, -%14, %18, %2\n\t"
        "v_fma_f32 %7, -%15, %19, %3\n\t"
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 1\n\t"
        "s_nop 1\n\t"
        "v_fma_f32 %0, -%12, %16, %0\n\t"
        "v_fma_f32 %1, -%13, %17, %1\n\t"
        "v_fma_f32 %2, -%14, %18, %2\n\t"
        "v_fma_f32 %3, -%15, %19, %3\n\t"
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0\n\t"
        "v_bfe_i32 %8, %4, 0, 1\n\t"
        "v_bfe_i32 %9, %5, 0, 1\n\t"
        "v_bfe_i32 %10, %6, 0, 1\n\t"
        "v_bfe_i32 %11, %7, 0, 1\n\t"
        "v_bfi_b32 %0, %8, %4, %0\n\t"
        "v_bfi_b32 %1, %9, %5, %1\n\t"
        "v_bfi_b32 %2, %10, %6, %2\n\t"
        "v_bfi_b32 %3, %11, %7, %3\n\t"
        "s_nop 1"
        : "+v"(na[0]), "+v"(na[1]), "+v"(na[2]), "+v"(na[3]),
          "=&v"(rd[0]), "=&v"(rd[1]), "=&v"(rd[2]), "=&v"(rd[3]),
          "=&v"(mask[0]), "=&v"(mask[1]), "=&v"(mask[2]), "=&v"(mask[3])
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]),
          "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]));
}

// Launches of at most a block a CU, one wave a SIMD.
constexpr unsigned kOneWaveBlocks = 256;

// The same for four outputs while round-down holds (between round_down and round_nearest): the
// rounding up is the negated rounding down of the negated sum, one instruction more a leaf and no
// mode switch, whose waits a single wave's four leaves cannot cover (8x4096x4096 on FP32 operands,
// 23 bits, one wave a SIMD: 367 us with rto_fnma4, 338 us so; 1000x768x3072, three blocks a
// CU, 375 and 403 us).
__device__ __forceinline__ void rto_fnma4_down(const float* a, const float* b, float* na) {
    float d[4], m[4];
    asm(
        "v_fma_f32 %4, -%12, %16, %0\n\t"
        "v_fma_f32 %5, -%13, %17, %1\n\t"
        "v_fma_f32 %6, -%14, %18, %2\n\t"
        "v_fma_f32 %7, -%15, %19, %3\n\t"
        "v_fma_f32 %0, %12, %16, -%0\n\t"
        "v_fma_f32 %1, %13, %17, -%1\n\t"
        "v_fma_f32 %2, %14, %18, -%2\n\t"
        "v_fma_f32 %3, %15, %19, -%3\n\t"
        "v_bfe_i32 %8, %4, 0, 1\n\t"
        "v_bfe_i32 %9, %5, 0, 1\n\t"
        "v_bfe_i32 %10, %6, 0, 1\n\t"
        "v_bfe_i32 %11, %7, 0, 1\n\t"
        "v_xor_b32 %0, 0x80000000, %0\n\t"
        "v_xor_b32 %1, 0x80000000, %1\n\t"
        "v_xor_b32 %2, 0x80000000, %2\n\t"
        "v_xor_b32 %3, 0x80000000, %3\n\t"
        "v_bfi_b32 %0, %8, %4, %0\n\t"
        "v_bfi_b32 %1, %9, %5, %1\n\t"
        "v_bfi_b32 %2, %10, %6, %2\n\t"
        "v_bfi_b32 %3, %11, %7, %3"
        : "+v"(na[0]), "+v"(na[1]), "+v"(na[2]), "+v"(na[3]),
          "=&v"(d[0]), "=&v"(d[1]), "=&v"(d[2]), "=&v"(d[3]),
          "=&v"(m[0]), "=&v"(m[1]), "=&v"(m[2]), "=&v"(m[3])
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]),
          "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]));
}
// Enter and leave round-down.  The accumulators pass through both statements, so nothing computed
// from them moves into the region.
__device__ __forceinline__ void round_down(float (&x)[4]) {
    asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 2\n\ts_nop 1"
                 : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]));
}
__device__ __forceinline__ void round_nearest(float (&x)[4]) {
    asm volatile("s_nop 1\n\ts_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0\n\ts_nop 1"
                 : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]));
}

// h <- binary16(h - a b), one rounding of the exact difference (see mix_fnma16), for the
// binary16 pairs h[i] = (h[2 i], h[2 i + 1]); the low halves first, so that no instruction follows
// the one that wrote half of its register.
__device__ __forceinline__ void mix_fnma_pairs16(const float* a, const float* b, uint32_t* h) {
    asm volatile(
        "v_fma_mixlo_f16 %0, -%8, %24, %0 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %1, -%10, %26, %1 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %2, -%12, %28, %2 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %3, -%14, %30, %3 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %4, -%16, %32, %4 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %5, -%18, %34, %5 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %6, -%20, %36, %6 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %7, -%22, %38, %7 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %0, -%9, %25, %0 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %1, -%11, %27, %1 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %2, -%13, %29, %2 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %3, -%15, %31, %3 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %4, -%17, %33, %4 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %5, -%19, %35, %5 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %6, -%21, %37, %6 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %7, -%23, %39, %7 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "s_nop 1"
        : "+v"(h[0]), "+v"(h[1]), "+v"(h[2]), "+v"(h[3]),
          "+v"(h[4]), "+v"(h[5]), "+v"(h[6]), "+v"(h[7])
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]),
          "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]),
          "v"(a[8]), "v"(a[9]), "v"(a[10]), "v"(a[11]),
          "v"(a[12]), "v"(a[13]), "v"(a[14]), "v"(a[15]),
          "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]),
          "v"(b[4]), "v"(b[5]), "v"(b[6]), "v"(b[7]),
          "v"(b[8]), "v"(b[9]), "v"(b[10]), "v"(b[11]),
          "v"(b[12]), "v"(b[13]), "v"(b[14]), "v"(b[15]));
}

__device__ __forceinline__ void mix_fnma_pairs4(const float* a, const float* b, uint32_t* h) {
    asm volatile(
        "v_fma_mixlo_f16 %0, -%2, %6, %0 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %1, -%4, %8, %1 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %0, -%3, %7, %0 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %1, -%5, %9, %1 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "s_nop 1"
        : "+v"(h[0]), "+v"(h[1])
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]),
          "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]));
}

// The same on one value a register (its low half), with the least magnitude of every result so far
// in `least`: mixed FMAs take 8 cycles a wave on gfx950, v_min_f16 2.5, v_min3_f16 over a pair 8.
__device__ __forceinline__ void mix_fnma16_least(const float* a, const float* b, uint32_t* u, uint32_t& least) {
    asm volatile(
        "v_fma_mixlo_f16 %0, -%17, %33, %0 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %1, -%18, %34, %1 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %2, -%19, %35, %2 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %3, -%20, %36, %3 op_sel_hi:[0,0,1]\n\t"
        "v_min_f16 %16, %16, |%0|\n\t"
        "v_fma_mixlo_f16 %4, -%21, %37, %4 op_sel_hi:[0,0,1]\n\t"
        "v_min_f16 %16, %16, |%1|\n\t"
        "v_fma_mixlo_f16 %5, -%22, %38, %5 op_sel_hi:[0,0,1]\n\t"
        "v_min_f16 %16, %16, |%2|\n\t"
        "v_fma_mixlo_f16 %6, -%23, %39, %6 op_sel_hi:[0,0,1]\n\t"
        "v_min_f16 %16, %16, |%3|\n\t"
        "v_fma_mixlo_f16 %7, -%24, %40, %7 op_sel_hi:[0,0,1]\n\t"
        "v_min_f16 %16, %16, |%4|\n\t"
        "v_fma_mixlo_f16 %8, -%25, %41, %8 op_sel_hi:[0,0,1]\n\t"
        "v_min_f16 %16, %16, |%5|\n\t"
        "v_fma_mixlo_f16 %9, -%26, %42, %9 op_sel_hi:[0,0,1]\n\t"
        "v_min_f16 %16, %16, |%6|\n\t"
        "v_fma_mixlo_f16 %10, -%27, %43, %10 op_sel_hi:[0,0,1]\n\t"
        "v_min_f16 %16, %16, |%7|\n\t"
        "v_fma_mixlo_f16 %11, -%28, %44, %11 op_sel_hi:[0,0,1]\n\t"
        "v_min_f16 %16, %16, |%8|\n\t"
        "v_fma_mixlo_f16 %12, -%29, %45, %12 op_sel_hi:[0,0,1]\n\t"
        "v_min_f16 %16, %16, |%9|\n\t"
        "v_fma_mixlo_f16 %13, -%30, %46, %13 op_sel_hi:[0,0,1]\n\t"
        "v_min_f16 %16, %16, |%10|\n\t"
        "v_fma_mixlo_f16 %14, -%31, %47, %14 op_sel_hi:[0,0,1]\n\t"
        "v_min_f16 %16, %16, |%11|\n\t"
        "v_fma_mixlo_f16 %15, -%32, %48, %15 op_sel_hi:[0,0,1]\n\t"
        "v_min_f16 %16, %16, |%12|\n\t"
        "v_min_f16 %16, %16, |%13|\n\t"
        "v_min_f16 %16, %16, |%14|\n\t"
        "v_min_f16 %16, %16, |%15|"
        : "+v"(u[0]), "+v"(u[1]), "+v"(u[2]), "+v"(u[3]),
          "+v"(u[4]), "+v"(u[5]), "+v"(u[6]), "+v"(u[7]),
          "+v"(u[8]), "+v"(u[9]), "+v"(u[10]), "+v"(u[11]),
          "+v"(u[12]), "+v"(u[13]), "+v"(u[14]), "+v"(u[15]), "+v"(least)
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]),
          "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]),
          "v"(a[8]), "v"(a[9]), "v"(a[10]), "v"(a[11]),
          "v"(a[12]), "v"(a[13]), "v"(a[14]), "v"(a[15]),
          "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]),
          "v"(b[4]), "v"(b[5]), "v"(b[6]), "v"(b[7]),
          "v"(b[8]), "v"(b[9]), "v"(b[10]), "v"(b[11]),
          "v"(b[12]), "v"(b[13]), "v"(b[14]), "v"(b[15]));
}

__device__ __forceinline__ void mix_fnma4_least(const float* a, const float* b, uint32_t* u, uint32_t& least) {
    asm volatile(
        "v_fma_mixlo_f16 %0, -%5, %9, %0 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %1, -%6, %10, %1 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %2, -%7, %11, %2 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %3, -%8, %12, %3 op_sel_hi:[0,0,1]\n\t"
        "s_nop 0\n\t"
        "v_min_f16 %4, %4, |%0|\n\t"
        "v_min_f16 %4, %4, |%1|\n\t"
        "v_min_f16 %4, %4, |%2|\n\t"
        "v_min_f16 %4, %4, |%3|"
        : "+v"(u[0]), "+v"(u[1]), "+v"(u[2]), "+v"(u[3]), "+v"(least)
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]),
          "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]));
}

// B of an implicit-GEMM convolution: a thread's four columns n = n0 + 4 * (tid % (BN / 4)) + j are
// the same in every slice (256 is a multiple of BN / 4); their output image, first input row
// and column and base offset are computed once.  A column past N gets a row that puts every
// tap outside the image.
template <int BN>
struct ConvCols {
    int ih0[4], iw0[4], base[4];
    __device__ __forceinline__ void init(const GemmArgs& g, int n0, int tid) {
        const ConvGeom& cv = g.cv;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int gn = n0 + 4 * (tid % (BN / 4)) + j;
            const uint32_t b = fast_div((uint32_t)gn, cv.div_pq);
            const uint32_t pq = (uint32_t)gn - b * cv.PQ;
            const uint32_t p = fast_div(pq, cv.div_q);
            const uint32_t q = pq - p * (uint32_t)cv.Q;
            const bool valid = gn < g.N;
            ih0[j] = valid ? (int)p * cv.sh - cv.ph : -(1 << 30);
            iw0[j] = (int)q * cv.sw - cv.pw;
            base[j] = valid ? (int)((int64_t)b * cv.sxb) + ih0[j] * cv.sxh + iw0[j] * cv.sxw : 0;
        }
    }
    // B(gk, n) of the four columns: the tap (c, r, s) of gk, zero in the padding and past K
    __device__ __forceinline__ float4 gather(const GemmArgs& g, int gk) const {
        const ConvGeom& cv = g.cv;
        const uint32_t d1 = fast_div((uint32_t)gk, cv.div_d1);
        const uint32_t rem = (uint32_t)gk - d1 * cv.D1;
        const uint32_t d2 = fast_div(rem, cv.div_d2);
        const uint32_t d3 = rem - d2 * (uint32_t)cv.D2;
        const int c = cv.krsc ? (int)d3 : (int)d1;
        const int r = cv.krsc ? (int)d1 : (int)d2;
        const int sx = cv.krsc ? (int)d2 : (int)d3;
        const int rr = r * cv.dh, ss = sx * cv.dw;
        const int koff = c * cv.sxc + rr * cv.sxh + ss * cv.sxw;
        float e[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int ih = ih0[j] + rr, iw = iw0[j] + ss;
            const bool in = gk < g.K && (unsigned)ih < (unsigned)cv.H &&
                            (unsigned)iw < (unsigned)cv.W;
            const float v = gld(g.B + (in ? base[j] + koff : 0));   // offset 0 when outside
            e[j] = in ? v : 0.0f;
        }
        return make_float4(e[0], e[1], e[2], e[3]);
    }
};

// Leading dimensions up to which a tile's offsets from its corner fit 32 bits (127 rows and a slice's
// 128 k).  With 64-bit offsets, held across the loop or recomputed for every slice, an
// 8192x4096x4096 training step at chunk 32 took 8.60 or 9.14 ms in place of 8.39.
constexpr int64_t kChainMaxLd = 1 << 25;

// Statistics of an operand slice (chunk 1, 23 bits): the largest magnitude and a lower bound on
// the exponent of every value's lowest set bit, as SliceStat's amax and key.
struct SliceKey {
    uint32_t amax = 0u, key = 0xFFFFFFFFu;
    __device__ __forceinline__ void add(float v) {
        const uint32_t b = __float_as_uint(v), sh = b << 1;
        amax = max(amax, sh);
        key = min(key, ((sh - 1u) >> 24) + min((uint32_t)__builtin_ctz(b | 0x80000000u), 24u));
    }
    __device__ __forceinline__ void add(const float4& v) { add(v.x); add(v.y); add(v.z); add(v.w); }
};

// The same of values stored as binary16 pairs, two at a time on the packed 16-bit units: the
// largest magnitude, and the least value of a lowest set bit, less one (x - (x with that bit
// cleared), exact in binary16; half of it for a power of two, whose pattern's lowest bit is the
// exponent's).  bad: a value that binary16 does not hold.
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
template <bool STAT>
struct PairKey {
    bool bad = false;
    u16x2 mx = {0, 0}, ls = {0xFFFF, 0xFFFF};
    __device__ __forceinline__ uint32_t add(float x, float y) {
        // truncation keeps a binary16 value
        const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(x, y));
        const f16x2 v = __builtin_bit_cast(f16x2, h);
        bad |= ((float)v.x != x) | ((float)v.y != y);
        if constexpr (STAT) {
            const u16x2 p = __builtin_bit_cast(u16x2, h & 0x7FFF7FFFu), one = {1, 1};
            const f16x2 d = __builtin_bit_cast(f16x2, p) - __builtin_bit_cast(f16x2, p & (p - one));
            mx = __builtin_elementwise_max(mx, p);
            ls = __builtin_elementwise_min(ls, __builtin_bit_cast(u16x2, d) - one);
        }
        return h;
    }
    // of both operands over the wave, valid in lane 63: {amax A, key A, amax B, key B} as SliceKey's
    static __device__ __forceinline__ uint4 wave(const PairKey& a, const PairKey& b) {
        auto least2 = [](u16x2 v) {
            return __builtin_bit_cast(u16x2, wave_last_u32(__builtin_bit_cast(uint32_t, v), ~0u, [](uint32_t x, uint32_t y) {
                return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, x),
                                                                              __builtin_bit_cast(u16x2, y)));
            }));
        };
        const u16x2 m = least2(~u16x2{max(a.mx.x, a.mx.y), max(b.mx.x, b.mx.y)});
        const u16x2 l = least2(u16x2{min(a.ls.x, a.ls.y), min(b.ls.x, b.ls.y)});
        auto bits = [](unsigned short x) {
            return __float_as_uint((float)__builtin_bit_cast(_Float16, x));
        };
        auto key = [&](unsigned short x) {
            return x == 0xFFFF ? 0xFFFFFFFFu : (bits((unsigned short)(x + 1)) >> 23) + 23u;
        };
        return make_uint4(bits((unsigned short)~m.x) << 1, key(l.x), bits((unsigned short)~m.y) << 1, key(l.y));
    }
};

// One BM x BN output tile; g.lda, g.ldb <= kChainMaxLd.
template <class T, int CHUNK, int KIND, bool CONV>
__device__ __forceinline__ void gemm_tile_chain(const GemmArgs& g, int tile_m, int tile_n, int tid,
                                                float* smem) {
    constexpr int BS = T::BS, BM = T::BM, BN = T::BN, BK = T::BK, NR = T::NR, KI = T::KI;
    constexpr int WMB = T::WMB, WNB = T::WNB;
    using LA = ChainLds<BM, BK, KI>;
    using LB = ChainLds<BN, BK, KI>;
    constexpr int NA4 = T::NA4, NB4 = T::NB4;
    // per-slice flags: an infinity or NaN among the operands (kChainMant, and any kind's chunk 1
    // but binary16's); a value that binary16 does not hold (binary16, chunk 1)
    constexpr bool kStep = CHUNK == 1;
    constexpr bool kF16Flag = kStep && KIND == kChainHalf;
    constexpr bool kFlag = KIND == kChainMant || kStep;
    // operand statistics: exact sums (23 bits), binary16's grid (10 bits)
    constexpr bool kStat = kStep && (KIND == kChainMant23 || KIND == kChainMant10);
    constexpr bool kWide = kStep && KIND == kChainMant10;   // a second flag: not binary16 operands
    // Chunk 1 without the matrix cores: a lane's outputs are SQ x SQ neighbours, SQ values of
    // each operand a k (an MFMA block's are 16 rows of one column, 17 values).  Kinds that
    // hold binary16 pairs also keep their slices as binary16 pairs while every value is one: half the
    // LDS bytes, no conversions, operands read as the packed FMA takes them.
    constexpr bool kOuter = kStep && KIND != kChainMant23;
    constexpr bool kPack = kStep && (KIND == kChainHalf || KIND == kChainMant10);
    constexpr int SQ = NR == 16 ? 4 : 2, SP = SQ / 2;
    constexpr int PGA = BM / 2 + 1, PGB = BN / 2 + 1;   // packed: uint4s per four k, one for the banks
    static_assert(!kStep || WMB * WNB == 1, "chunk 1: one block a wave");
    static_assert(4 * PGA * (BK / 4) <= LA::FLOATS && 4 * PGB * (BK / 4) <= LB::FLOATS, "packed slices fit");
    static_assert(kStep || (CHUNK >= KI && BK % CHUNK == 0),
                  "whole MFMAs per chunk, whole chunks per slice");
    constexpr float kPadA = kStep ? 0.0f : -0.0f;   // k past K, see the head comment
    using vec = typename std::conditional<BS == 32, f32x16, f32x4>::type;

    const int lane = tid & 63, wave = tid >> 6;
    const int lcol = lane % BS, lhi = lane / BS;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int am0 = (wave / T::WC) * BS * WMB, bn0 = (wave % T::WC) * BS * WNB;
    uint32_t* flags = (uint32_t*)(smem + 2 * T::BUF_FLOATS);
    uint32_t* stats = flags + 4;   // [buffer][wave][amax A, key A, amax B, key B]

    // Element mapping: float4 f = tid + 256 * it of the A slice is row m = f / (BK / 4),
    // k = 4 * (f % (BK / 4)) .. + 3 of a row-major A, or k = f / (BM / 4), m = 4 * (f % (BM / 4))
    // .. + 3 of a transposed one; likewise B.  Offsets are from the tile's corner.  They are
    // recomputed for every slice from a copy of tid that the compiler cannot see through:
    // held across the loop, they and the edges' element offsets spill.
    // kPack: row-major rows come in neighbouring pairs (it, it + 1), a packed store each.
    auto otid = [&]() { int t = tid; asm volatile("" : "+v"(t)); return t; };
    auto rows_of = [](int t) { return kPack ? t / (BK / 4) * 2 : t / (BK / 4); };
    auto rows_step = [](int it) { return kPack ? (it & 1) + (it >> 1) * (2048 / BK) : it * (1024 / BK); };
    ConvCols<BN> cols;
    if constexpr (CONV) cols.init(g, n0, tid);
    const float* A0 = g.A + (g.ta ? (int64_t)m0 : (int64_t)m0 * g.lda);
    const float* B0 = g.B + (g.tb ? (int64_t)n0 * g.ldb : (int64_t)n0);

    // NV float4s of an operand slice: R rows (A's m, B's n), `left` of them inside the matrix from
    // the tile's corner p on, kl k left in K.  kmaj: stored k-major (four rows per float4).
    // Inside the matrix a thread's float4s lie a wave-uniform step apart (256 float4s are
    // whole rows), from an offset that is computed once.
    auto load_op = [&](auto& v, auto rows, const float* p, bool kmaj, int64_t ld, int left, int kl,
                       float pad) {
        constexpr int R = decltype(rows)::value, NV = R * BK / 1024;
        if (kl >= BK && left >= R) {
            const uint32_t o = kmaj ? (uint32_t)(tid / (R / 4)) * (uint32_t)ld + (uint32_t)(4 * (tid % (R / 4)))
                                    : (uint32_t)rows_of(tid) * (uint32_t)ld + (uint32_t)(4 * (tid % (BK / 4)));
#pragma unroll
            for (int it = 0; it < NV; ++it)
                v[it] = gld4u(p + (kmaj ? it * (1024 / R) : rows_step(it)) * ld + o);
            return;
        }
        const int t = otid();   // an edge: elements from clamped addresses, `pad` past K
#pragma unroll
        for (int it = 0; it < NV; ++it) {
            float e[4];
            if (kmaj) {
                const int c = 4 * (t % (R / 4)), k = t / (R / 4) + it * (1024 / R);
                const uint32_t o = (uint32_t)min(k, kl - 1) * (uint32_t)ld;
                if (c + 3 < left) {
                    v[it] = gld4u(p + (o + (uint32_t)c));
                    if (k >= kl) v[it] = make_float4(pad, pad, pad, pad);
                    continue;
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    e[j] = gld(p + (o + (uint32_t)min(c + j, left - 1)));
                    e[j] = k < kl ? e[j] : pad;
                }
            } else {
                const int k = 4 * (t % (BK / 4));
                const int r = min(rows_of(t) + rows_step(it), left - 1);
                const uint32_t o = (uint32_t)r * (uint32_t)ld;
                if (kl >= BK) {
                    v[it] = gld4u(p + (o + (uint32_t)k));
                    continue;
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    e[j] = gld(p + (o + (uint32_t)min(k + j, kl - 1)));
                    e[j] = k + j < kl ? e[j] : pad;
                }
            }
            v[it] = make_float4(e[0], e[1], e[2], e[3]);
        }
    };
    float4 va[NA4], vb[NB4];
    auto load_slice = [&](int k0) {
        const int kl = g.K - k0;
        load_op(va, std::integral_constant<int, BM>{}, A0 + (g.ta ? (int64_t)k0 * g.lda : (int64_t)k0),
                g.ta != 0, g.lda, g.M - m0, kl, kPadA);
        if constexpr (CONV) {
            const int t = otid();
#pragma unroll
            for (int it = 0; it < NB4; ++it)
                vb[it] = cols.gather(g, k0 + t / (BN / 4) + it * (1024 / BN));
        } else {
            load_op(vb, std::integral_constant<int, BN>{},
                    B0 + (g.tb ? (int64_t)k0 : (int64_t)k0 * g.ldb), g.tb == 0, g.ldb, g.N - n0, kl,
                    0.0f);
        }
    };
    // registers -> LDS buffer, as FP32 or as binary16 pairs
    using Pairs = PairKey<kStat>;
    auto put_slice = [&](int buf, bool packed, Pairs& ka, Pairs& kb) {
        float* As = smem + buf * T::BUF_FLOATS;
        auto put = [&](float* S, auto lds, auto rows, const auto& v, bool kmaj, Pairs& key) {
            using L = decltype(lds);
            constexpr int R = decltype(rows)::value, NV = R * BK / 1024, PG = R / 2 + 1;
            if (kPack && packed) {   // [k / 4][row pair][k % 4]
                auto pk = [&](float x, float y) { return key.add(x, y); };
                if (kmaj) {
                    const int k = tid / (R / 4);
                    uint32_t* d = (uint32_t*)S + (k >> 2) * 4 * PG + 8 * (tid % (R / 4)) + (k & 3);
#pragma unroll
                    for (int it = 0; it < NV; ++it) {
                        d[it * (256 / R) * 4 * PG] = pk(v[it].x, v[it].y);
                        d[it * (256 / R) * 4 * PG + 4] = pk(v[it].z, v[it].w);
                    }
                } else {
                    uint4* d = (uint4*)S + (tid % (BK / 4)) * PG + tid / (BK / 4);
#pragma unroll
                    for (int it = 0; it + 1 < NV; it += 2)
                        d[it * (512 / BK)] = make_uint4(pk(v[it].x, v[it + 1].x), pk(v[it].y, v[it + 1].y),
                                                        pk(v[it].z, v[it + 1].z), pk(v[it].w, v[it + 1].w));
                }
                return;
            }
            if (kmaj) {   // float4 `it` lies 1024 / R (a multiple of 4) k further
                const int k = tid / (R / 4);
                float* d = S + L::row(k) + ((4 * (tid % (R / 4))) ^ L::swz(k));
#pragma unroll
                for (int it = 0; it < NV; ++it) *(float4*)(d + it * (256 / R) * L::GROUP) = v[it];
            } else {      // 4 k of a row, 1024 / BK (at most 32) rows further each time
                // The thread's own row, below that step, shares no bit with it or with the swizzle
                // (a multiple of 32 where the step is 32 rows, of 16 where it is 16 or 8): it is added.
                float* d = S + (tid % (BK / 4)) * L::GROUP + (kPack ? 0 : tid / (BK / 4));
#pragma unroll
                for (int it = 0; it < NV; ++it) {
                    const int r = (kPack ? rows_of(tid) : 0) + rows_step(it);
                    d[0 * R + (r ^ L::swz(0))] = v[it].x;
                    d[1 * R + (r ^ L::swz(1))] = v[it].y;
                    d[2 * R + (r ^ L::swz(2))] = v[it].z;
                    d[3 * R + (r ^ L::swz(3))] = v[it].w;
                }
            }
        };
        put(As, LA{}, std::integral_constant<int, BM>{}, va, g.ta != 0, ka);
        put(As + LA::FLOATS, LB{}, std::integral_constant<int, BN>{}, vb, CONV || g.tb == 0, kb);
    };
    // Statistics that cannot help are not taken: after a slice whose products alone are too wide
    // for exact sums or the grid, the next ones (1, 3, 7, then 15 in turn, for as long as they stay
    // so) are stored without them (a 2048x1024x4096 training step on FP32 operands, 23 bits: 2.77 ->
    // 2.45 ms; 4096^3 on FP32 operands, 10 bits: 7.34 -> 7.08 ms).
    int skip = 0, last_skip = 0;
    auto judge = [&](bool hopeless) {
        last_skip = hopeless ? min(2 * last_skip + 1, 15) : 0;
        skip = last_skip;
    };
    // fl: the slice's flags; full: with every statistic (else 10 bits' largest magnitudes and a
    // bound on B's exponents only)
    auto store_slice = [&](int buf, int fl, bool packed, bool full) {
        Pairs pa, pb;
        put_slice(buf, packed, pa, pb);
        if (kPack && packed) {
            bool bad = pa.bad | pb.bad;
            if constexpr (kStat) {
                const u16x2 m = __builtin_elementwise_max(pa.mx, pb.mx);
                bad |= max(m.x, m.y) >= 0x7C00;   // an infinity
                const uint4 w = Pairs::wave(pa, pb);
                if (lane == 63) *(uint4*)(stats + buf * 16 + wave * 4) = w;
            }
            if (bad) flags[fl + (kStat ? 40 : 0)] = 1u;
            return;
        }
        SliceKey ka, kb;
        auto over = [](const auto& v, auto f) {
            bool any = false;
#pragma unroll
            for (int it = 0; it < (int)(sizeof(v) / sizeof(float4)); ++it)
                any |= f(v[it].x) | f(v[it].y) | f(v[it].z) | f(v[it].w);
            return any;
        };
        auto not16 = [](float x) { return (float)(_Float16)x != x; };
        if constexpr (kF16Flag) {
            if (over(va, not16) | over(vb, not16)) flags[fl] = 1u;
        } else if constexpr (kFlag) {
            float z = 0.0f;   // 0 * v summed: NaN as soon as one v is not finite
            auto sum = [&](float x) { z = __builtin_fmaf(x, 0.0f, z); return false; };
            over(va, sum);
            over(vb, sum);
            if (z != 0.0f) flags[fl] = 1u;   // z is +-0 or NaN
        }
        if (!full) {
            if constexpr (kWide) {
                uint32_t ma = 0u, mb = 0u, nb = ~0u;
                over(va, [&](float x) { ma = max(ma, __float_as_uint(x) << 1); return false; });
                over(vb, [&](float x) {
                    const uint32_t b = __float_as_uint(x) << 1;
                    mb = max(mb, b);
                    nb = min(nb, b - 1u);
                    return false;
                });
                ma = wave_max_u32(ma);
                mb = wave_max_u32(mb);
                nb = wave_min_u32(nb) >> 24;   // the least exponent of B's values, in place of the lowest bit's
                if (lane == 63)
                    *(uint4*)(stats + buf * 16 + wave * 4) = make_uint4(ma, 0u, mb, nb == 0u ? 1u : nb + 23u);
            }
            return;
        }
        if constexpr (kWide) {   // A binary16 values, B of at most 11 significant bits
            if (over(va, not16) | over(vb, [](float x) { return (__float_as_uint(x) & 0x1FFFu) != 0u; }))
                flags[fl + 36] = 1u;
        }
        if constexpr (kStat) {
#pragma unroll
            for (int it = 0; it < NA4; ++it) ka.add(va[it]);
#pragma unroll
            for (int it = 0; it < NB4; ++it) kb.add(vb[it]);
            const uint4 w = make_uint4(wave_max_u32(ka.amax), wave_min_u32(ka.key),
                                       wave_max_u32(kb.amax), wave_min_u32(kb.key));
            if (lane == 63) *(uint4*)(stats + buf * 16 + wave * 4) = w;
        }
    };

    // the accumulators; kNeg: negated, from -0 (binary16, and every kind's chunk 1)
    constexpr bool kNeg = KIND == kChainHalf || kStep;
    float acc[WMB][WNB][NR];
#pragma unroll
    for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
        for (int bj = 0; bj < WNB; ++bj)
#pragma unroll
            for (int r = 0; r < NR; ++r) acc[bi][bj][r] = kNeg ? -0.0f : 0.0f;

    // rows and columns of the matrix from this wave's corner on
    const int rows_in = g.M - m0 - __builtin_amdgcn_readfirstlane(am0);
    const int cols_in = g.N - n0 - __builtin_amdgcn_readfirstlane(bn0);
    const bool wave_in = rows_in > 0 && cols_in > 0;

    // Leaves in pieces of PN outputs.  PIPE: a chunk's leaves run between the next chunk's
    // MFMAs, from its second step on (the first piece still waits for the sums to settle), so
    // one wave keeps both the matrix cores and the VALU busy; the leaf before the first chunk
    // works on zero sums, which leave zero accumulators as they are.  The wide tile (64 sums a
    // wave) has no registers for a second set.
    constexpr int STEPS = kStep ? 1 : CHUNK / KI;
    constexpr int PN = NR == 4 ? 4 : 8, PIECES = WMB * WNB * NR / PN;
    constexpr bool PIPE = STEPS >= 2 && WMB * WNB * NR <= 32;
    constexpr int FIRST = STEPS >= 4 ? 1 : 0;
    constexpr int PER = PIPE ? (PIECES + STEPS - 2 - FIRST) / (STEPS - 1 - FIRST) : 0;
    auto piece = [&](vec (&sums)[WMB][WNB], int n, bool spec) {
        const int blk = n / (NR / PN), o0 = n % (NR / PN) * PN;
        const int bi = blk / WNB, bj = blk % WNB;
        float p[PN], x[PN];
#pragma unroll
        for (int r = 0; r < PN; ++r) {
            p[r] = sums[bi][bj][o0 + r];
            x[r] = acc[bi][bj][o0 + r];
        }
        chain_leaves<KIND, PN>(p, x, spec, g, [&](int o) {   // the lowest row of output o0 + o
            const int row = bi * BS + ((o0 + o) >> 2) * 8 + ((o0 + o) & 3);
            return row < rows_in && bj * BS < cols_in;
        });
#pragma unroll
        for (int r = 0; r < PN; ++r) acc[bi][bj][o0 + r] = x[r];
    };
    auto settle = [&](vec (&v)[WMB][WNB]) {
        if constexpr (WMB * WNB == 4) mfma_settle(v[0][0], v[0][1], v[1][0], v[1][1]);
        else if constexpr (WNB == 2) mfma_settle(v[0][0], v[0][1]);
        else if constexpr (WMB == 2) mfma_settle(v[0][0], v[1][0]);
        else mfma_settle(v[0][0]);
    };
    vec prev[WMB][WNB];
    bool sprev = false;
    if constexpr (PIPE) {
#pragma unroll
        for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
            for (int bj = 0; bj < WNB; ++bj)
#pragma unroll
                for (int r = 0; r < NR; ++r) prev[bi][bj][r] = 0.0f;
    }
    // this lane's part of its operand reads' addresses: row lhi of a step's k, swizzled column
    int ra[WMB], rb[WNB];
#pragma unroll
    for (int bi = 0; bi < WMB; ++bi)
        ra[bi] = lhi * BM + ((am0 + bi * BS + lcol) ^ LA::swz(lhi));
#pragma unroll
    for (int bj = 0; bj < WNB; ++bj)
        rb[bj] = lhi * BN + ((bn0 + bj * BS + lcol) ^ LB::swz(lhi));

    // ---- chunk 1: every k's leaf, on the negated accumulators
    // This lane's outputs: r is row out_row(r), column out_col(r) of the wave's block.
    const int orow = kOuter ? SQ * (lane >> 3) : lhi * 4, ocol = kOuter ? SQ * (lane & 7) : lcol;
    auto out_row = [&](int r) { return orow + (kOuter ? r % SQ : (r >> 2) * 8 + (r & 3)); };
    auto out_col = [&](int r) { return ocol + (kOuter ? r / SQ : 0); };
    // operand values of output r, as the leaves take them
    auto ax = [](int r) { return kOuter ? r % SQ : r; };
    auto bx = [](int r) { return kOuter ? r / SQ : 0; };
    constexpr int NA = kOuter ? SQ : NR, NB = kOuter ? SQ : 1;
    auto fetch_k = [&](const float* Ap, const float* Bp, int k, float* a, float* b) {
        auto quads = [](float* o, const float* p) {
            const float4 v = *(const float4*)p;
            o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
        };
        auto pair = [](float* o, const float* p) {
            const float2 v = *(const float2*)p;
            o[0] = v.x; o[1] = v.y;
        };
        const float* ap = Ap + LA::row(k);
        const float* bp = Bp + LB::row(k) + ((bn0 + ocol) ^ LB::swz(k));
        if constexpr (kOuter) {
            ap += (am0 + orow) ^ LA::swz(k);
            if constexpr (SQ == 4) {
                quads(a, ap);
                quads(b, bp);
            } else {
                pair(a, ap);
                pair(b, bp);
            }
        } else {
#pragma unroll
            for (int rq = 0; rq < NR / 4; ++rq)
                quads(a + 4 * rq, ap + ((am0 + rq * 8 + orow) ^ LA::swz(k)));
            b[0] = *bp;
        }
    };
    // leaf(a, b), a[NA] and b[NB], for every k < kmax, in groups of four k (those past K add -0):
    // a group's next k is read while the current one computes
    auto for_k32 = [&](const float* As, const float* Bs, int kmax, auto leaf) {
        float a[2][NA], b[2][NB];
        constexpr bool kAhead = NR == 4;
        if constexpr (kAhead) fetch_k(As, Bs, 0, a[0], b[0]);
        const int ng = (kmax + 3) / 4;
        for (int q = 0; q < ng; ++q) {
            const float* Aq = As + q * LA::GROUP;
            const float* Bq = Bs + q * LB::GROUP;
            const int adv = q + 1 < ng ? 1 : 0;   // the last group reads its own first k again
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (!kAhead) fetch_k(Aq, Bq, j, a[j & 1], b[j & 1]);
                else if (j < 3) fetch_k(Aq, Bq, j + 1, a[(j + 1) & 1], b[(j + 1) & 1]);
                else fetch_k(Aq + adv * LA::GROUP, Bq + adv * LB::GROUP, 0, a[0], b[0]);
                leaf(a[j & 1], b[j & 1]);
            }
        }
    };
    // A packed slice's pairs of four k: group q of this lane's rows (columns), pair p, k % 4 = j is
    // component j of [p].  leaf(a, b) for every group; ahead: the next one read while it computes,
    // groups in twos (a slice is padded to its full length).
    auto for_k16 = [&](auto ahead, const float* As, const float* Bs, int kmax, auto leaf) {
        const uint4* Ap = (const uint4*)As + (am0 + orow) / 2;
        const uint4* Bp = (const uint4*)Bs + (bn0 + ocol) / 2;
        uint4 a[2][SP], b[2][SP];
        auto fetch = [&](int set, int q) {
#pragma unroll
            for (int p = 0; p < SP; ++p) {
                a[set][p] = Ap[q * PGA + p];
                b[set][p] = Bp[q * PGB + p];
            }
        };
        if constexpr (!ahead.value) {
            for (int q = 0; q < (kmax + 3) / 4; ++q) {
                fetch(0, q);
                leaf(a[0], b[0]);
            }
            return;
        }
        const int ng = (kmax + 7) / 8 * 2;
        fetch(0, 0);
        for (int q = 0; q < ng; q += 2) {
            fetch(1, q + 1);
            leaf(a[0], b[0]);
            fetch(0, q + 2 < ng ? q + 2 : q);
            leaf(a[1], b[1]);
        }
    };
    auto word = [](const uint4& v, int j) { return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w; };
    auto pair_of = [&](const uint4& v, int j) { return __builtin_bit_cast(f16x2, word(v, j)); };
    // for_k32 over either form of slice
    auto for_k = [&](bool packed, const float* As, const float* Bs, int kmax, auto leaf) {
        if constexpr (kPack) {
            if (packed) {
                for_k16(std::false_type{}, As, Bs, kmax, [&](const uint4* a4, const uint4* b4) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        float a[SQ], b[SQ];
#pragma unroll
                        for (int p = 0; p < SP; ++p) {
                            a[2 * p] = (float)pair_of(a4[p], j).x;
                            a[2 * p + 1] = (float)pair_of(a4[p], j).y;
                            b[2 * p] = (float)pair_of(b4[p], j).x;
                            b[2 * p + 1] = (float)pair_of(b4[p], j).y;
                        }
                        leaf(a, b);
                    }
                });
                return;
            }
        }
        for_k32(As, Bs, kmax, leaf);
    };
    // The general leaf over a slice, out of line per leaf: slices with an infinity or a NaN, and
    // binary16 sums that reach 65520 (or held values that are not binary16).
    auto general_slice = [&](bool packed, const float* As, const float* Bs, int kmax) {
        const LeafGen L = leaf_gen(g);
        auto at = [&](const float* S, auto lds, int pg, int k, int row) -> float {
            if (kPack && packed)
                return (float)((const _Float16*)S)[((k >> 2) * pg + row / 2) * 8 + (k & 3) * 2 + row % 2];
            using L = decltype(lds);
            return S[L::row(k) + (row ^ L::swz(k))];
        };
        for (int k = 0; k < kmax; ++k)
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const float a = at(As, LA{}, PGA, k, am0 + out_row(r)), b = at(Bs, LB{}, PGB, k, bn0 + out_col(r));
                float& na = acc[0][0][r];
                na = -(float)leaf_slow<LeafGen>((double)a * (double)b, -(double)na, L);
            }
    };
    // While `held`, the accumulators are binary16 pairs scaled by 2^hs (exact both ways where
    // they are used), in the first half of acc's registers.
    bool held = false;
    int hs = 0;
    float acc_bound = 0.0f;   // 10 bits, held: above every accumulator of the wave
    int accL = 1000;   // 23 and 10 bits: every accumulator of the wave is a multiple of 2^accL
    auto get_held = [&](uint32_t (&h)[NR / 2]) {
#pragma unroll
        for (int r = 0; r < NR / 2; ++r) h[r] = __float_as_uint(acc[0][0][r]);
    };
    auto put_held = [&](const uint32_t (&h)[NR / 2]) {
#pragma unroll
        for (int r = 0; r < NR; ++r) acc[0][0][r] = r < NR / 2 ? __uint_as_float(h[r]) : 0.0f;
    };
    auto hold = [&](int to) {
        hs = to;
        uint32_t h[NR / 2];
#pragma unroll
        for (int r = 0; r < NR / 2; ++r)
            h[r] = __builtin_bit_cast(uint32_t, f16x2{(_Float16)__builtin_ldexpf(acc[0][0][2 * r], hs),
                                                      (_Float16)__builtin_ldexpf(acc[0][0][2 * r + 1], hs)});
        put_held(h);
        held = true;
    };
    auto unhold = [&]() {
        uint32_t h[NR / 2];
        get_held(h);
#pragma unroll
        for (int r = 0; r < NR / 2; ++r) {
            const f16x2 v = __builtin_bit_cast(f16x2, h[r]);
            acc[0][0][2 * r] = __builtin_ldexpf((float)v.x, -hs);
            acc[0][0][2 * r + 1] = __builtin_ldexpf((float)v.y, -hs);
        }
        held = false;
    };
    // a leaf's operands per output, for the assembly
    auto spread = [&](const float* a, const float* b, float (&av)[NR], float (&bv)[NR]) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            av[r] = a[ax(r)];
            bv[r] = b[bx(r)];
        }
    };
    // every leaf by directed roundings
    auto directed = [&](bool packed, const float* As, const float* Bs, int kmax) {
        float (&x)[NR] = acc[0][0];
        auto leaf = [&](auto down, const float* a, const float* b) {
            float av[NR], bv[NR];
            spread(a, b, av, bv);
            if constexpr (NR == 16) rto_fnma16(av, bv, x);
            else if constexpr (down.value) rto_fnma4_down(av, bv, x);
            else rto_fnma4(av, bv, x);
            if constexpr (KIND != kChainMant23)
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    const uint32_t t = __float_as_uint(x[r]);
                    x[r] = __uint_as_float((t + g.dr_half + __builtin_amdgcn_ubfe(t, g.dr_rf, 1u)) &
                                           g.dr_mask);
                }
        };
        if constexpr (NR == 4) {
            if (gridDim.x <= kOneWaveBlocks) {
                round_down(x);
                for_k(packed, As, Bs, kmax, [&](const float* a, const float* b) { leaf(std::true_type{}, a, b); });
                round_nearest(x);
                return;
            }
        }
        for_k(packed, As, Bs, kmax, [&](const float* a, const float* b) { leaf(std::false_type{}, a, b); });
    };
    // the packed binary16 leaves of a packed slice, B scaled by 2^hs where `scaled`
    auto packed_leaves = [&](const float* As, const float* Bs, int kmax, auto scaled) {
        const _Float16 sc = (_Float16)__builtin_ldexpf(1.0f, hs);
        uint32_t hp[NR / 2];
        get_held(hp);
        for_k16(std::true_type{}, As, Bs, kmax, [&](const uint4* a4, const uint4* b4) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int c = 0; c < SQ; ++c) {
                    f16x2 b = pair_of(b4[c / 2], j);
                    if constexpr (scaled.value) b = b * f16x2{sc, sc};
                    b = c & 1 ? f16x2{b.y, b.y} : f16x2{b.x, b.x};
#pragma unroll
                    for (int p = 0; p < SP; ++p)
                        hp[c * SP + p] = __builtin_bit_cast(
                            uint32_t, __builtin_elementwise_fma(-pair_of(a4[p], j), b,
                                                                __builtin_bit_cast(f16x2, hp[c * SP + p])));
                }
        });
        put_held(hp);
    };
    // the same from an FP32 slice of binary16 values (scaled: B of binary16's significand)
    auto packed_leaves32 = [&](const float* As, const float* Bs, int kmax) {
        uint32_t hp[NR / 2];
        get_held(hp);
        for_k32(As, Bs, kmax, [&](const float* a, const float* b) {
#pragma unroll
            for (int c = 0; c < SQ; ++c) {
                const _Float16 bv = (_Float16)__builtin_ldexpf(b[c], hs);
#pragma unroll
                for (int p = 0; p < SP; ++p) {
                    const f16x2 av = {(_Float16)a[2 * p], (_Float16)a[2 * p + 1]};
                    hp[c * SP + p] = __builtin_bit_cast(
                        uint32_t, __builtin_elementwise_fma(-av, f16x2{bv, bv},
                                                            __builtin_bit_cast(f16x2, hp[c * SP + p])));
                }
            }
        });
        put_held(hp);
    };
    auto step_slice = [&](bool packed, const float* As, const float* Bs, int kmax, bool special,
                          bool wide16, bool full, int buf) {
        if constexpr (KIND == kChainHalf) {
            // Held as binary16 pairs while every accumulator is a binary16 value below 2^15 at a
            // slice's start.  The binary16 FMA (operands binary16 too: packed, two leaves an
            // instruction) and the mixed one round the exact h - a b once, which is the leaf as long
            // as no result passes 65504; an infinity or NaN stays one, so one look at the slice's
            // end finds it, and the slice is redone from its start values.
            if (!held) {
                bool ok = true;
#pragma unroll
                for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
                    for (int bj = 0; bj < WNB; ++bj)
#pragma unroll
                        for (int r = 0; r < NR; ++r) {
                            const float x = acc[bi][bj][r];
                            ok &= (float)(_Float16)x == x && fabsf(x) < 32768.0f;
                        }
                if (!wave_in || __all(ok)) hold(0);
            }
            if (held) {
                uint32_t h0[NR / 2], h[NR / 2];
                get_held(h0);
                if (packed) {
                    packed_leaves(As, Bs, kmax, std::false_type{});
                } else if (!special) {
                    packed_leaves32(As, Bs, kmax);
                } else {
                    get_held(h);
                    for_k32(As, Bs, kmax, [&](const float* a, const float* b) {
                        float av[NR], bv[NR];
                        spread(a, b, av, bv);
                        if constexpr (NR == 16) mix_fnma_pairs16(av, bv, h);
                        else mix_fnma_pairs4(av, bv, h);
                    });
                    put_held(h);
                }
                get_held(h);
                bool over = false;
#pragma unroll
                for (int r = 0; r < NR / 2; ++r) {
                    const uint32_t e = ~h[r];   // exponent all ones: inf or NaN
                    over |= (e & 0x7C00u) == 0u || (e & 0x7C000000u) == 0u;
                }
                if (wave_in && __any(over)) {
                    put_held(h0);
                    unhold();
                }
            }
            if (__builtin_expect(!held, 0)) general_slice(packed, As, Bs, kmax);
        } else {
            if (__builtin_expect(special, 0)) {
                if (KIND == kChainMant10 && held) unhold();
                general_slice(packed, As, Bs, kmax);
                accL = -1000;
                return;
            }
            if constexpr (KIND == kChainMant23) {
                // Exact sums: when every sum of 32 consecutive k is exact in FP32, each leaf is the
                // plain FMA (RTO24 and the rounding keep an exact sum), and 32 of them are 32 / KI
                // steps of the f32 MFMA on the negated accumulator, whose round-to-nearest zeros
                // are the negated RTO24 zeros.  All sums are multiples of 2^L, L the lower of the
                // products' lowest bit (from the slice's statistics) and the accumulators', and
                // below 2^S with 2^S > |acc| + 33 amax_A amax_B: exact when S <= L + 24.
                if (!full) {
                    accL = -1000;
                    directed(false, As, Bs, kmax);
                    return;
                }
                uint32_t amA = 0u, amB = 0u, kyA = ~0u, kyB = ~0u;
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint4 v = *(const uint4*)(stats + buf * 16 + w * 4);
                    amA = max(amA, v.x); kyA = min(kyA, v.y);
                    amB = max(amB, v.z); kyB = min(kyB, v.w);
                }
                const int sL = amA == 0u || amB == 0u ? 1000 : (int)kyA + (int)kyB - 300;
                // an upper bound on a product's magnitude, at least 2^-126
                const float pm = fmaxf(__uint_as_float(amA >> 1) * __uint_as_float(amB >> 1), 0x1p-126f) *
                                 1.0000152587890625f;
                judge(__builtin_amdgcn_readfirstlane((int)(__float_as_uint(pm) >> 23)) - 126 >
                      __builtin_amdgcn_readfirstlane(sL) + 24);
                for (int kq = 0; kq < kmax; kq += 32) {
                    float am = 0.0f;
#pragma unroll
                    for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
                        for (int bj = 0; bj < WNB; ++bj)
#pragma unroll
                            for (int r = 0; r < NR; ++r) am = fmaxf(am, fabsf(acc[bi][bj][r]));
                    const float bnd = __builtin_fmaf(33.0f, pm, am) * 1.0000152587890625f;
                    const int S = (int)(__float_as_uint(bnd) >> 23) - 126;
                    bool ok = S <= 127 && sL >= -149 && __all(S <= sL + 24);
                    if (ok && accL < sL) {   // unknown or finer: the accumulators' own lowest bit
                        if (accL == -1000) {
                            uint32_t key = ~0u;
#pragma unroll
                            for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
                                for (int bj = 0; bj < WNB; ++bj)
#pragma unroll
                                    for (int r = 0; r < NR; ++r) {
                                        const uint32_t x = __float_as_uint(acc[bi][bj][r]);
                                        key = min(key, (((x << 1) - 1u) >> 24) +
                                                           min((uint32_t)__builtin_ctz(x | 0x80000000u), 24u));
                                    }
                            key = wave_min_u32(key);
                            accL = (int)__builtin_amdgcn_readlane((int)key, 63) - 150;   // 129 for zeros
                        }
                        ok = accL >= -149 && __all(S <= min(sL, accL) + 24);
                    }
                    const float* Aq = As + kq / 4 * LA::GROUP;
                    const float* Bq = Bs + kq / 4 * LB::GROUP;
                    if (ok) {
                        accL = min(accL, sL);
                        vec c[WMB][WNB];
#pragma unroll
                        for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
                            for (int bj = 0; bj < WNB; ++bj)
#pragma unroll
                                for (int r = 0; r < NR; ++r) c[bi][bj][r] = acc[bi][bj][r];
#pragma unroll
                        for (int i = 0; i < 32 / KI; ++i) {
                            float a[WMB], b[WNB];
#pragma unroll
                            for (int bi = 0; bi < WMB; ++bi) a[bi] = -Aq[LA::row(KI * i) + ra[bi]];
#pragma unroll
                            for (int bj = 0; bj < WNB; ++bj) b[bj] = Bq[LB::row(KI * i) + rb[bj]];
#pragma unroll
                            for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
                                for (int bj = 0; bj < WNB; ++bj) {
                                    if constexpr (BS == 32)
                                        c[bi][bj] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                                            a[bi], b[bj], c[bi][bj], 0, 0, 0);
                                    else
                                        c[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                            a[bi], b[bj], c[bi][bj], 0, 0, 0);
                                }
                        }
                        settle(c);
#pragma unroll
                        for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
                            for (int bj = 0; bj < WNB; ++bj)
#pragma unroll
                                for (int r = 0; r < NR; ++r) acc[bi][bj][r] = c[bi][bj][r];
                    } else {
                        accL = -1000;
                        directed(false, Aq, Bq, min(32, kmax - kq));
                    }
                }
            } else if constexpr (KIND == kChainMant10) {
                // 10 bits: binary16's significand, any exponent.  Held as binary16 values scaled by
                // 2^hs, hs the same for the wave: below 2^15, and from 2^-14 up, binary16 rounds a
                // sum as the accumulator does.  Below 2^-14 it does too where every sum is a
                // multiple of 2^-24 scaled (then it has at most 10 bits there); elsewhere the least
                // result tells: above 2^-14, no sum was below.  Bounds per 32 k, for the wave: sums
                // are below 2^S > (1 + 2^-11)^32 (|acc| + 33 amax_A amax_B), and multiples of 2^L as
                // for exact sums (a rounding keeps a coarser or equal grid).
                uint32_t amA = 0u, amB = 0u, kyA = ~0u, kyB = ~0u;
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint4 v = *(const uint4*)(stats + buf * 16 + w * 4);
                    amA = max(amA, v.x); kyA = min(kyA, v.y);
                    amB = max(amB, v.z); kyB = min(kyB, v.w);
                }
                const bool zero = amA == 0u || amB == 0u;
                const int sL = !full ? -1000 : zero ? 1000 : (int)kyA + (int)kyB - 300;
                const int bLsb = amB == 0u ? 1000 : (int)kyB - 150;
                const int bTop = amB == 0u ? -1000 : (int)(amB >> 24) - 127;
                const float pm = fmaxf(__uint_as_float(amA >> 1) * __uint_as_float(amB >> 1), 0x1p-126f) *
                                 1.0000152587890625f;
                if (full && !packed)
                    judge(wide16 || __builtin_amdgcn_readfirstlane((int)(__float_as_uint(pm) >> 23)) - 126 >
                                        __builtin_amdgcn_readfirstlane(sL) + 39);
                auto held_leaves = [&](const float* Aq, const float* Bq, int kn) {
                    if (!packed) packed_leaves32(Aq, Bq, kn);
                    else if (hs == 0) packed_leaves(Aq, Bq, kn, std::false_type{});
                    else packed_leaves(Aq, Bq, kn, std::true_type{});
                };
                for (int kq = 0; kq < kmax; kq += 32) {
                    const float* Aq = As + kq / 4 * (packed ? 4 * PGA : LA::GROUP);
                    const float* Bq = Bs + kq / 4 * (packed ? 4 * PGB : LB::GROUP);
                    const int kn = min(32, kmax - kq);
                    // Held already: a bound carried from one 32 k to the next, no look at the values.
                    if (held) {
                        const float bnd = __builtin_fmaf(33.0f, pm, acc_bound) * 1.0158f;   // 1.015749...
                        const int S = __builtin_amdgcn_readfirstlane((int)(__float_as_uint(bnd) >> 23)) - 126;
                        if (!wide16 && S <= 15 - hs && S <= 127 && bTop <= 15 - hs &&
                            min(sL, bLsb) >= -24 - hs && sL >= -126) {
                            accL = min(accL, sL);
                            acc_bound = bnd;
                            held_leaves(Aq, Bq, kn);
                            continue;
                        }
                        unhold();
                    }
                    // the wave's largest and smallest accumulator magnitudes
                    float hi_f = 0.0f, lo_f = 0x1.fffffep+127f;
#pragma unroll
                    for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
                        for (int bj = 0; bj < WNB; ++bj)
#pragma unroll
                            for (int r = 0; r < NR; ++r) {
                                hi_f = fmaxf(hi_f, fabsf(acc[bi][bj][r]));
                                lo_f = fminf(lo_f, fabsf(acc[bi][bj][r]));
                            }
                    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane(
                        (int)wave_max_u32(__float_as_uint(hi_f)), 63);
                    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane(
                        (int)wave_min_u32(__float_as_uint(lo_f)), 63);
                    const float bnd = __builtin_fmaf(33.0f, pm, __uint_as_float(hi)) * 1.0158f;   // 1.015749...
                    const int S = (int)(__float_as_uint(bnd) >> 23) - 126;
                    const bool in = S <= 127;   // finite, and no overflow rule
                    bool grid = in && !wide16 && sL >= -126 && S - sL <= 39;
                    if (grid && accL == -1000) {   // unknown: the accumulators' own lowest bit
                        uint32_t key = ~0u;
#pragma unroll
                        for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
                            for (int bj = 0; bj < WNB; ++bj)
#pragma unroll
                                for (int r = 0; r < NR; ++r) {
                                    const uint32_t x = __float_as_uint(acc[bi][bj][r]);
                                    key = min(key, (((x << 1) - 1u) >> 24) +
                                                       min((uint32_t)__builtin_ctz(x | 0x80000000u), 24u));
                                }
                        accL = __builtin_amdgcn_readlane((int)wave_min_u32(key), 63) - 150;   // 129 for zeros
                    }
                    const int L = min(sL, accL);
                    // hs for the grid: 2^L to 2^-24 or above, 2^S to 2^15 or below, B within binary16
                    const int gLo = max(-24 - L, -24 - bLsb), gHi = min(15 - S, 15 - bTop);
                    grid = grid && L >= -126 && gLo <= gHi && (!packed || (gLo <= 15 && gHi >= -24));
                    if (grid) {
                        accL = L;
                        // none where it can be, else in the middle, so that it lasts; itself a
                        // binary16 value where a packed B is scaled
                        const int mid = gLo <= 0 && gHi >= 0 ? 0 : (gLo + gHi) >> 1;
                        hold(packed ? max(min(mid, 15), -24) : mid);
                        acc_bound = bnd;
                        held_leaves(Aq, Bq, kn);
                        continue;
                    }
                    accL = -1000;
                    // checked: the smallest start value at 2^-14 or above scaled (so that all convert),
                    // sums below 2^-126 seen too (hs <= 112), b 2^hs FP32-normal
                    const int eLo = (int)(lo >> 23) - 127;
                    const int cLo = max(-14 - eLo, -126 - bLsb), cHi = min(min(15 - S, 112), 126 - bTop);
                    if (in && lo != 0u && cLo <= cHi) {
                        uint32_t u[NR], least = 0x7BFFu;
#pragma unroll
                        for (int r = 0; r < NR; ++r)
                            u[r] = __builtin_bit_cast(uint16_t, (_Float16)__builtin_ldexpf(acc[0][0][r], cHi));
                        for_k(packed, Aq, Bq, kn, [&](const float* a, const float* b) {
                            float bs[NB], av[NR], bv[NR];
#pragma unroll
                            for (int c = 0; c < NB; ++c) bs[c] = __builtin_ldexpf(b[c], cHi);
                            spread(a, bs, av, bv);
                            if constexpr (NR == 16) mix_fnma16_least(av, bv, u, least);
                            else mix_fnma4_least(av, bv, u, least);
                        });
                        if (__all((least & 0xFFFFu) > 0x0400u)) {   // 2^-14
#pragma unroll
                            for (int r = 0; r < NR; ++r)
                                acc[0][0][r] = __builtin_ldexpf(
                                    (float)__builtin_bit_cast(_Float16, (uint16_t)u[r]), -cHi);
                            continue;
                        }
                    }
                    directed(packed, Aq, Bq, kn);
                }
            } else {
                directed(false, As, Bs, kmax);
            }
        }
    };

    // Non-finite flags, three in turn: slice s reads flag s % 3 between its barrier and the next;
    // meanwhile the store of slice s + 1 sets flag (s + 1) % 3 and flag (s + 2) % 3 (read last by
    // slice s - 1, before this slice's barrier) is cleared for slice s + 2.
    if constexpr (kFlag) {
        if (tid < 3) flags[tid] = flags[tid + 36] = flags[tid + 40] = 0u;
        lds_barrier();
    }
    // Slices are stored packed until one does not fit: that one is stored again, from the registers
    // that still hold it, and the tile's others as FP32.
    bool packed = kPack;
    bool full = true;   // slice k0's statistics
    int fs = 0, buf = 1;
    for (int k0 = -BK; k0 < g.K; k0 += BK) {   // the first pass only loads slice 0
        bool special = false, wide16 = false;
        if (k0 >= 0) lds_barrier();   // slice k0 is in buffer buf; the other one is free
        const int fn = k0 < 0 ? 0 : fs == 2 ? 0 : fs + 1;
        if constexpr (kFlag) {
            if (k0 >= 0) {
                auto flag = [&](int i) { return __builtin_amdgcn_readfirstlane((int)flags[fs + i]) != 0; };
                if (kPack && packed) {
                    packed = !flag(kStat ? 40 : 0);
                    if (!packed) {   // (no other slice's flags are set or read here)
                        store_slice(buf, fs, false, true);
                        lds_barrier();
                    }
                }
                special = flag(0);
                if constexpr (kWide) wide16 = flag(36);
                if (tid == 0) {
                    const int fc = fn == 2 ? 0 : fn + 1;
                    flags[fc] = 0u;
                    if constexpr (kWide) flags[fc + 36] = flags[fc + 40] = 0u;
                }
            }
        }
        const bool has_next = k0 + BK < g.K;
        if (has_next) load_slice(k0 + BK);   // in flight while this slice computes
        const float* As = smem + buf * T::BUF_FLOATS;
        const float* Bs = As + LA::FLOATS;
        if constexpr (kStep) {
            if (k0 >= 0) step_slice(packed, As, Bs, min(BK, g.K - k0), special, wide16, full, buf);
        }
        // chunks that hold a k < K (none in the first pass)
        const int nq = kStep || k0 < 0 ? 0 : min(BK, g.K - k0 + CHUNK - 1) / CHUNK;
        for (int q = 0; q < nq; ++q) {
            const int kb = q * CHUNK;
            // The chunk's k in groups of G MFMA steps (64 cycles of the matrix cores each group):
            // the next group's LDS reads are issued before the current group's MFMAs, which
            // with the other waves' cover their latency.
            constexpr int G = BS == 32 || STEPS < 2 ? 1 : 2, NG = STEPS / G;
            float a[2][G][WMB], b[2][G][WNB];
            auto fetch = [&](int set, int grp) {
#pragma unroll
                for (int i = 0; i < G; ++i) {
                    const int k = kb + KI * (grp * G + i);   // lane row k + lhi: no carry past k | (KI - 1)
#pragma unroll
                    for (int bi = 0; bi < WMB; ++bi) a[set][i][bi] = As[LA::row(k) + ra[bi]];
#pragma unroll
                    for (int bj = 0; bj < WNB; ++bj) b[set][i][bj] = Bs[LB::row(k) + rb[bj]];
                }
            };
            fetch(0, 0);
            vec part[WMB][WNB];
#pragma unroll
            for (int grp = 0; grp < NG; ++grp) {
                if (grp + 1 < NG) fetch((grp + 1) & 1, grp + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < G; ++i) {
                    const int step = grp * G + i;
#pragma unroll
                    for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
                        for (int bj = 0; bj < WNB; ++bj) {
                            vec c;
                            if (step == 0) {
#pragma unroll
                                for (int r = 0; r < NR; ++r) c[r] = 0.0f;
                            } else {
                                c = part[bi][bj];
                            }
                            vec d;
                            if constexpr (BS == 32)
                                d = __builtin_amdgcn_mfma_f32_32x32x2f32(a[grp & 1][i][bi],
                                                                         b[grp & 1][i][bj], c, 0, 0, 0);
                            else
                                d = __builtin_amdgcn_mfma_f32_16x16x4f32(a[grp & 1][i][bi],
                                                                         b[grp & 1][i][bj], c, 0, 0, 0);
                            if (PIPE && step == STEPS - 1) prev[bi][bj] = d;
                            else part[bi][bj] = d;
                        }
                    if constexpr (PIPE) {   // leaf pieces of the previous chunk
                        if (step >= FIRST && step < STEPS - 1) {
                            __builtin_amdgcn_sched_barrier(0);
                            if (step == FIRST) settle(prev);
#pragma unroll
                            for (int n = 0; n < PER; ++n)
                                if ((step - FIRST) * PER + n < PIECES)
                                    piece(prev, (step - FIRST) * PER + n, sprev);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (PIPE) {
                sprev = special;
            } else {
                settle(part);
#pragma unroll
                for (int n = 0; n < PIECES; ++n) piece(part, n, special);
            }
        }
        buf ^= 1;
        if (has_next) {
            full = skip == 0;
            skip = full ? 0 : skip - 1;
            store_slice(buf, fn, packed, full);
        }
        fs = fn;
    }
    if constexpr (PIPE) {   // the last chunk's leaves
        settle(prev);
#pragma unroll
        for (int n = 0; n < PIECES; ++n) piece(prev, n, sprev);
    }

    if constexpr (kPack)
        if (held) unhold();
    // epilogue (cutlass LinearCombination): D = alpha * acc, or fma(alpha, acc, beta * C);
    // a convolution's D(m, n) / C(m, n) sit at b * sdb + m * sdm + (p * Q + q) * sdpq
#pragma unroll
    for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
        for (int bj = 0; bj < WNB; ++bj) {
            int64_t col = 0;
            const int64_t row_stride_d = CONV ? g.cv.sdm : g.ldd, row_stride_c = CONV ? g.cv.sdm : g.ldc;
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const int gn = n0 + bn0 + bj * BS + out_col(r);
                if (r == 0 || out_col(r) != out_col(r - 1)) {
                    col = gn;
                    if constexpr (CONV) {
                        const uint32_t b = fast_div((uint32_t)gn, g.cv.div_pq);
                        col = (int64_t)b * g.cv.sdb + (int64_t)((uint32_t)gn - b * g.cv.PQ) * g.cv.sdpq;
                    }
                }
                const int gm = m0 + am0 + bi * BS + out_row(r);
                if (gm >= g.M || gn >= g.N) continue;
                const float a = kNeg ? -acc[bi][bj][r] : acc[bi][bj][r];
                float d;
                if (g.beta != 0.0f)
                    d = __builtin_fmaf(g.alpha, a, g.beta * gld(g.C + (int64_t)gm * row_stride_c + col));
                else
                    d = g.alpha * a;
                gst(g.D + (int64_t)gm * row_stride_d + col, d);
            }
        }
}

}  // namespace lofamd
