// lof_gemm_chain.hpp -- emulated-accumulation GEMM tile for chunks of 2 to 32, with every chunk
// sum on the f32 matrix cores (gfx950).
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
enum ChainKind : int { kChainMant = 0, kChainMant23 = 1, kChainHalf = 2 };

// An operand slice in LDS: R rows (A's m, B's n) by BK k, k-major in groups of four k that
// start PAD floats apart, the row swizzled by k.  An MFMA operand read takes KI consecutive k of
// 64 / KI consecutive rows each; the swizzle puts them in different banks (64 banks of 4
// bytes), and PAD spreads the transposing stores of a row-major operand, whose lanes hold
// consecutive groups of four k.  (Rows of R + 4 floats: every operand read had two-way conflicts.)
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
    static constexpr int SMEM_FLOATS = 2 * BUF_FLOATS + 4;   // + 3 non-finite flags
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
template <int KIND, int NR>
__device__ __forceinline__ void chain_leaves(float (&p)[NR], float (&acc)[NR], bool special,
                                             const GemmArgs& g) {
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
                if (fabsf(t[o]) >= g.half_top) t[o] = chain_half_slow(p[o], acc[o], leaf_gen(g));
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

// One BM x BN output tile of chunk sums of CHUNK (2..32) products; g.lda, g.ldb <= kChainMaxLd.
constexpr int64_t kChainMaxLd = 1 << 22;   // a tile's offsets from its corner fit 32 bits

template <class T, int CHUNK, int KIND, bool CONV>
__device__ __forceinline__ void gemm_tile_chain(const GemmArgs& g, int tile_m, int tile_n, int tid,
                                                float* smem) {
    constexpr int BS = T::BS, BM = T::BM, BN = T::BN, BK = T::BK, NR = T::NR, KI = T::KI;
    constexpr int WMB = T::WMB, WNB = T::WNB;
    using LA = ChainLds<BM, BK, KI>;
    using LB = ChainLds<BN, BK, KI>;
    constexpr int NA4 = T::NA4, NB4 = T::NB4;
    constexpr bool kFlag = KIND == kChainMant;
    static_assert(CHUNK >= KI && BK % CHUNK == 0, "whole MFMAs per chunk, whole chunks per slice");
    using vec = typename std::conditional<BS == 32, f32x16, f32x4>::type;

    const int lane = tid & 63, wave = tid >> 6;
    const int lcol = lane % BS, lhi = lane / BS;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int am0 = (wave / T::WC) * BS * WMB, bn0 = (wave % T::WC) * BS * WNB;
    uint32_t* flags = (uint32_t*)(smem + 2 * T::BUF_FLOATS);

    // Element mapping: float4 f = tid + 256 * it of the A slice is row m = f / (BK / 4),
    // k = 4 * (f % (BK / 4)) .. + 3 of a row-major A, or k = f / (BM / 4), m = 4 * (f % (BM / 4))
    // .. + 3 of a transposed one; likewise B.  Offsets are from the tile's corner.  They are
    // recomputed for every slice from a copy of tid that the compiler cannot see through:
    // held across the loop, they and the edges' element offsets spill.
    auto otid = [&]() { int t = tid; asm volatile("" : "+v"(t)); return t; };
    ConvCols<BN> cols;
    if constexpr (CONV) cols.init(g, n0, tid);
    const float* A0 = g.A + (g.ta ? (int64_t)m0 : (int64_t)m0 * g.lda);
    const float* B0 = g.B + (g.tb ? (int64_t)n0 * g.ldb : (int64_t)n0);

    // NV float4s of an operand slice: R rows (A's m, B's n), `left` of them inside the matrix from
    // the tile's corner p on, kl k left in K.  kmaj: stored k-major (four rows per float4).
    // Inside the matrix a thread's float4s lie a wave-uniform step apart (256 float4s are
    // whole rows), so each load is one offset register and a scalar base.
    auto load_op = [&](auto& v, auto rows, const float* p, bool kmaj, int64_t ld, int left, int kl,
                       float pad) {
        constexpr int R = decltype(rows)::value, NV = R * BK / 1024;
        if (kl >= BK && left >= R) {
            const uint32_t o = kmaj ? (uint32_t)(tid / (R / 4)) * (uint32_t)ld + (uint32_t)(4 * (tid % (R / 4)))
                                    : (uint32_t)(tid / (BK / 4)) * (uint32_t)ld + (uint32_t)(4 * (tid % (BK / 4)));
            const int64_t step = (kmaj ? 1024 / R : 1024 / BK) * ld;
#pragma unroll
            for (int it = 0; it < NV; ++it) v[it] = gld4u(p + it * step + o);
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
                const int r = min(t / (BK / 4) + it * (1024 / BK), left - 1);
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
                g.ta != 0, g.lda, g.M - m0, kl, -0.0f);
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
    // registers -> LDS buffer; fl: the slice's non-finite flag
    auto store_slice = [&](int buf, int fl) {
        float* As = smem + buf * T::BUF_FLOATS;
        float z = 0.0f;   // 0 * v summed: NaN as soon as one v is not finite
        auto put = [&](float* S, auto lds, auto rows, const auto& v, bool kmaj) {
            using L = decltype(lds);
            constexpr int R = decltype(rows)::value, NV = R * BK / 1024;
            if (kmaj) {   // float4 `it` lies 1024 / R (a multiple of 4) k further
                const int k = tid / (R / 4);
                float* d = S + L::row(k) + ((4 * (tid % (R / 4))) ^ L::swz(k));
#pragma unroll
                for (int it = 0; it < NV; ++it) *(float4*)(d + it * (256 / R) * L::GROUP) = v[it];
            } else {      // 4 k of a row, 1024 / BK (at most 32) rows further each time
                float* d = S + (tid % (BK / 4)) * L::GROUP + tid / (BK / 4);
#pragma unroll
                for (int it = 0; it < NV; ++it) {
                    const int r = it * (1024 / BK);
                    d[0 * R + (r ^ L::swz(0))] = v[it].x;
                    d[1 * R + (r ^ L::swz(1))] = v[it].y;
                    d[2 * R + (r ^ L::swz(2))] = v[it].z;
                    d[3 * R + (r ^ L::swz(3))] = v[it].w;
                }
            }
            if constexpr (kFlag) {
#pragma unroll
                for (int it = 0; it < NV; ++it) {
                    z = __builtin_fmaf(v[it].x, 0.0f, z);
                    z = __builtin_fmaf(v[it].y, 0.0f, z);
                    z = __builtin_fmaf(v[it].z, 0.0f, z);
                    z = __builtin_fmaf(v[it].w, 0.0f, z);
                }
            }
        };
        put(As, LA{}, std::integral_constant<int, BM>{}, va, g.ta != 0);
        put(As + LA::FLOATS, LB{}, std::integral_constant<int, BN>{}, vb, CONV || g.tb == 0);
        if constexpr (kFlag)
            if (z != 0.0f) flags[fl] = 1u;   // z is +-0 or NaN
    };

    float acc[WMB][WNB][NR];   // kChainHalf: -acc, from -0
#pragma unroll
    for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
        for (int bj = 0; bj < WNB; ++bj)
#pragma unroll
            for (int r = 0; r < NR; ++r) acc[bi][bj][r] = KIND == kChainHalf ? -0.0f : 0.0f;

    // Leaves in pieces of PN outputs.  PIPE: a chunk's leaves run between the next chunk's
    // MFMAs, from its second step on (the first piece still waits for the sums to settle), so
    // one wave keeps both the matrix cores and the VALU busy; the leaf before the first chunk
    // works on zero sums, which leave zero accumulators as they are.  The wide tile (64 sums a
    // wave) has no registers for a second set.
    constexpr int STEPS = CHUNK / KI;
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
        chain_leaves<KIND, PN>(p, x, spec, g);
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

    // Non-finite flags, three in turn: slice s reads flag s % 3 between its barrier and the next;
    // meanwhile the store of slice s + 1 sets flag (s + 1) % 3 and flag (s + 2) % 3 (read last by
    // slice s - 1, before this slice's barrier) is cleared for slice s + 2.
    if constexpr (kFlag) {
        if (tid < 3) flags[tid] = 0u;
        lds_barrier();
    }
    int fs = 0, buf = 1;
    for (int k0 = -BK; k0 < g.K; k0 += BK) {   // the first pass only loads slice 0
        bool special = false;
        if (k0 >= 0) lds_barrier();   // slice k0 is in buffer buf; the other one is free
        const int fn = k0 < 0 ? 0 : fs == 2 ? 0 : fs + 1;
        if constexpr (kFlag) {
            if (k0 >= 0) {
                special = __builtin_amdgcn_readfirstlane((int)flags[fs]) != 0;
                if (tid == 0) flags[fn == 2 ? 0 : fn + 1] = 0u;
            }
        }
        const bool has_next = k0 + BK < g.K;
        if (has_next) load_slice(k0 + BK);   // in flight while this slice computes
        const float* As = smem + buf * T::BUF_FLOATS;
        const float* Bs = As + LA::FLOATS;
        // chunks that hold a k < K (none in the first pass)
        const int nq = k0 < 0 ? 0 : min(BK, g.K - k0 + CHUNK - 1) / CHUNK;
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
        if (has_next) store_slice(buf, fn);
        fs = fn;
    }
    if constexpr (PIPE) {   // the last chunk's leaves
        settle(prev);
#pragma unroll
        for (int n = 0; n < PIECES; ++n) piece(prev, n, sprev);
    }

    // epilogue (cutlass LinearCombination): D = alpha * acc, or fma(alpha, acc, beta * C);
    // a convolution's D(m, n) / C(m, n) sit at b * sdb + m * sdm + (p * Q + q) * sdpq
#pragma unroll
    for (int bi = 0; bi < WMB; ++bi)
#pragma unroll
        for (int bj = 0; bj < WNB; ++bj) {
            const int gn = n0 + bn0 + bj * BS + lcol;
            int64_t col = gn, row_stride_d = g.ldd, row_stride_c = g.ldc;
            if constexpr (CONV) {
                const uint32_t b = fast_div((uint32_t)gn, g.cv.div_pq);
                col = (int64_t)b * g.cv.sdb + (int64_t)((uint32_t)gn - b * g.cv.PQ) * g.cv.sdpq;
                row_stride_d = row_stride_c = g.cv.sdm;
            }
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const int gm = m0 + am0 + bi * BS + (r >> 2) * 8 + lhi * 4 + (r & 3);
                if (gm >= g.M || gn >= g.N) continue;
                const float a = KIND == kChainHalf ? -acc[bi][bj][r] : acc[bi][bj][r];
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
