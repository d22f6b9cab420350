// lof_gemm_few.hpp -- emulated-accumulation GEMM tile for products with few outputs (gfx950):
// 16 x 16 outputs a workgroup, one a lane, for the accumulators and chunks of lof_gemm_chain.hpp.
//
// An output is a serial chain over K.  With few outputs a SIMD holds one wave, which issues an
// instruction every 5 cycles however long its dependency chain is: the time is K times the
// instructions a wave issues per k, so each lane takes one output and as many SIMDs as there are
// get a wave.  (The matrix cores' blocks put 4 or 16 outputs in a lane, on a quarter of the waves.)
// Chunk sums are then plain FMAs, four chunks' chains interleaved.
//
// Operand slices of 128 k sit row by row in double-buffered LDS (rows of 132 floats: the 16 columns
// a wave reads 16 bytes of are in different banks), loaded two slices ahead: 4 KB a wave in flight
// is what covers the memory's latency at one wave a SIMD.
//
// 8x4096x4096, us on the 16x64 tile of lof_gemm_chain.hpp and here: e4m3 operands, chunk 1, 23 bits
// 141 and 74, 10 bits 161 and 100, binary16-shaped 114 and 60, chunk 8 129 and 50; FP32 operands, chunk 1, 23
// bits 305 and 88, 7 bits 368 and 101; chunk 32, 23 bits 83 and 55.
#pragma once

#include "lof_gemm_chain.hpp"

namespace lofamd {

constexpr int kFewB = 16, kFewK = 128, kFewRow = kFewK + 4;
constexpr int kFewBuf = 2 * kFewB * kFewRow;
constexpr int kFewSmem = 2 * kFewBuf + 36;   // + 3 flags, statistics

// Four chunk leaves in turn, acc <- round(RTO24(acc + p)), in one statement so that nothing else runs
// in round-down.  The rounding up is the negated rounding down of the negated sum; the odd of
// the two is RTO24's result, the rounded-down one where both are even (an exact sum, or -0).
#define LOF_FEW_LEAF(P)                                                                          \
    "v_add_f32 %1, %0, " P "\n\t"                                                               \
    "v_sub_f32 %2, -%0, " P "\n\t"                                                              \
    "v_bfe_i32 %3, %2, 0, 1\n\t"                                                                \
    "v_xor_b32 %2, 0x80000000, %2\n\t"                                                          \
    "v_bfi_b32 %0, %3, %2, %1\n\t"
#define LOF_FEW_ROUND                                                                            \
    "v_bfe_u32 %3, %0, %8, 1\n\t"                                                               \
    "v_add3_u32 %0, %0, %9, %3\n\t"                                                             \
    "v_and_b32 %0, %10, %0\n\t"
#define LOF_FEW_DOWN "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 2\n\ts_nop 1\n\t"
#define LOF_FEW_NEAREST "s_nop 1\n\ts_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0\n\ts_nop 1"

template <int KIND>
__device__ __forceinline__ void few_add4(const float (&p)[4], float& acc, const GemmArgs& g) {
    float d, t, m;
    if constexpr (KIND == kChainMant23)
        asm volatile(LOF_FEW_DOWN LOF_FEW_LEAF("%4") LOF_FEW_LEAF("%5") LOF_FEW_LEAF("%6")
                         LOF_FEW_LEAF("%7") LOF_FEW_NEAREST
                     : "+v"(acc), "=&v"(d), "=&v"(t), "=&v"(m)
                     : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]));
    else
        asm volatile(LOF_FEW_DOWN LOF_FEW_LEAF("%4") LOF_FEW_ROUND LOF_FEW_LEAF("%5") LOF_FEW_ROUND
                         LOF_FEW_LEAF("%6") LOF_FEW_ROUND LOF_FEW_LEAF("%7") LOF_FEW_ROUND LOF_FEW_NEAREST
                     : "+v"(acc), "=&v"(d), "=&v"(t), "=&v"(m)
                     : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "s"(g.dr_rf), "s"(g.dr_half),
                       "s"(g.dr_mask));
}

// Chunk 1, four k in turn on the negated accumulator (see rto_fnma4_down), while round-down holds.
#define LOF_FEW_STEP(A, B)                                                                       \
    "v_fma_f32 %1, -" A ", " B ", %0\n\t"                                                       \
    "v_fma_f32 %2, " A ", " B ", -%0\n\t"                                                       \
    "v_bfe_i32 %3, %1, 0, 1\n\t"                                                                \
    "v_xor_b32 %2, 0x80000000, %2\n\t"                                                          \
    "v_bfi_b32 %0, %3, %1, %2\n\t"
#define LOF_FEW_STEP_ROUND                                                                       \
    "v_bfe_u32 %3, %0, %12, 1\n\t"                                                              \
    "v_add3_u32 %0, %0, %13, %3\n\t"                                                            \
    "v_and_b32 %0, %14, %0\n\t"

template <int KIND>
__device__ __forceinline__ void few_fnma4_down(const float4& a, const float4& b, float& na, const GemmArgs& g) {
    float d, t, m;
    if constexpr (KIND == kChainMant23)
        asm(LOF_FEW_STEP("%4", "%8") LOF_FEW_STEP("%5", "%9") LOF_FEW_STEP("%6", "%10") LOF_FEW_STEP("%7", "%11")
            : "+v"(na), "=&v"(d), "=&v"(t), "=&v"(m)
            : "v"(a.x), "v"(a.y), "v"(a.z), "v"(a.w), "v"(b.x), "v"(b.y), "v"(b.z), "v"(b.w));
    else
        asm(LOF_FEW_STEP("%4", "%8") LOF_FEW_STEP_ROUND LOF_FEW_STEP("%5", "%9") LOF_FEW_STEP_ROUND
                LOF_FEW_STEP("%6", "%10") LOF_FEW_STEP_ROUND LOF_FEW_STEP("%7", "%11") LOF_FEW_STEP_ROUND
            : "+v"(na), "=&v"(d), "=&v"(t), "=&v"(m)
            : "v"(a.x), "v"(a.y), "v"(a.z), "v"(a.w), "v"(b.x), "v"(b.y), "v"(b.z), "v"(b.w),
              "s"(g.dr_rf), "s"(g.dr_half), "s"(g.dr_mask));
}

// h <- binary16(h - a b) for four k in turn (see mix_fnma_pairs16); the second form keeps the least
// magnitude of the results.  A wait state after each result that is half a register.
__device__ __forceinline__ void few_mix4(const float4& a, const float4& b, uint32_t& h) {
    asm("v_fma_mixlo_f16 %0, -%1, %5, %0 op_sel_hi:[0,0,1]\n\t"
        "s_nop 0\n\t"
        "v_fma_mixlo_f16 %0, -%2, %6, %0 op_sel_hi:[0,0,1]\n\t"
        "s_nop 0\n\t"
        "v_fma_mixlo_f16 %0, -%3, %7, %0 op_sel_hi:[0,0,1]\n\t"
        "s_nop 0\n\t"
        "v_fma_mixlo_f16 %0, -%4, %8, %0 op_sel_hi:[0,0,1]\n\t"
        "s_nop 0"
        : "+v"(h)
        : "v"(a.x), "v"(a.y), "v"(a.z), "v"(a.w), "v"(b.x), "v"(b.y), "v"(b.z), "v"(b.w));
}
__device__ __forceinline__ void few_mix4_least(const float4& a, const float4& b, uint32_t& h, uint32_t& least) {
    asm("v_fma_mixlo_f16 %0, -%2, %6, %0 op_sel_hi:[0,0,1]\n\t"
        "s_nop 0\n\t"
        "v_min_f16 %1, %1, |%0|\n\t"
        "v_fma_mixlo_f16 %0, -%3, %7, %0 op_sel_hi:[0,0,1]\n\t"
        "s_nop 0\n\t"
        "v_min_f16 %1, %1, |%0|\n\t"
        "v_fma_mixlo_f16 %0, -%4, %8, %0 op_sel_hi:[0,0,1]\n\t"
        "s_nop 0\n\t"
        "v_min_f16 %1, %1, |%0|\n\t"
        "v_fma_mixlo_f16 %0, -%5, %9, %0 op_sel_hi:[0,0,1]\n\t"
        "s_nop 0\n\t"
        "v_min_f16 %1, %1, |%0|\n\t"
        "s_nop 0"
        : "+v"(h), "+v"(least)
        : "v"(a.x), "v"(a.y), "v"(a.z), "v"(a.w), "v"(b.x), "v"(b.y), "v"(b.z), "v"(b.w));
}

// Products the tile takes: 16-byte loads need four k of a row-major operand, four rows of a k-major
// one.
inline bool few_takes(int64_t M, int64_t N, int64_t K, bool ta, bool tb) {
    return K >= 4 && (!ta || M >= 4) && (tb || N >= 4);
}

// One 16 x 16 output tile (few_takes), for any leading dimensions.
template <int CHUNK, int KIND>
__device__ __forceinline__ void gemm_tile_few(const GemmArgs& g, int tile_m, int tile_n, int tid, float* smem) {
    constexpr int BK = kFewK, ROW = kFewRow;
    constexpr bool kStep = CHUNK == 1;
    constexpr bool kFlag = KIND == kChainMant || (kStep && KIND != kChainHalf);
    constexpr bool kStat = kStep && (KIND == kChainMant23 || KIND == kChainMant10);
    constexpr float kPadA = kStep ? 0.0f : -0.0f;   // k past K, as in gemm_tile_chain
    const int lane = tid & 63, wave = tid >> 6;
    const int row = tid / kFewB, colm = tid % kFewB;
    const int m0 = tile_m * kFewB, n0 = tile_n * kFewB;
    // A wave past the matrix's rows repeats its last one; its outputs are dropped and take no general
    // leaves.
    const bool wave_in = m0 + 4 * __builtin_amdgcn_readfirstlane(wave) < g.M;
    uint32_t* flags = (uint32_t*)(smem + 2 * kFewBuf);
    uint32_t* stats = flags + 4;   // [buffer][wave][amax A, key A, amax B, key B]
    const float* A0 = g.A + (g.ta ? (int64_t)m0 : (int64_t)m0 * g.lda);
    const float* B0 = g.B + (g.tb ? (int64_t)n0 * g.ldb : (int64_t)n0);

    // Two float4s a thread and operand: 4 k of row f / 32, or 4 rows of k = f / 4 where the operand
    // is stored k-major.  Every load is unconditional, at an address moved back inside the matrix
    // at its edges (hence 4 rows or k at least, few_takes): behind a branch the compiler could
    // not count the loads in flight and would wait for all of them.  The last slices are loaded
    // again where there is none to come.
    const int last = (g.K - 1) / BK * BK;
    auto load_op = [&](float4 (&v)[2], const float* p, bool kmaj, int64_t ld, int left, int kl) {
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const int f = tid + 256 * it;
            const int r = kmaj ? min(f >> 2, kl - 1) : min(f >> 5, left - 1);
            const int c = kmaj ? min(4 * (f & 3), left - 4) : min(4 * (f & 31), kl - 4);
            v[it] = gld4u(p + ((int64_t)r * ld + c));
        }
    };
    float4 va[2][2], vb[2][2];   // slices in flight, by parity
    auto load_slice = [&](auto set, int k) {
        const int k0 = min(k, last), kl = g.K - k0;
        load_op(va[set.value], A0 + (g.ta ? (int64_t)k0 * g.lda : (int64_t)k0), g.ta != 0, g.lda, g.M - m0, kl);
        load_op(vb[set.value], B0 + (g.tb ? (int64_t)k0 : (int64_t)k0 * g.ldb), g.tb == 0, g.ldb, g.N - n0, kl);
    };
    // what load_op moved back at an edge in its place, `pad` past K (rows past the matrix: any)
    auto mend_op = [&](float4 (&v)[2], bool kmaj, int left, int kl, float pad) {
        if (kl >= BK && left >= kFewB) return;
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const int f = tid + 256 * it;
            const int c = kmaj ? 4 * (f & 3) : 4 * (f & 31), n = kmaj ? left : kl;
            const int sh = min(c - min(c, n - 4), 3);
            const float4 x = v[it];
            float4 y = sh == 0 ? x : sh == 1 ? make_float4(x.y, x.z, x.w, x.w)
                     : sh == 2 ? make_float4(x.z, x.w, x.w, x.w) : make_float4(x.w, x.w, x.w, x.w);
            if (kmaj) {
                if ((f >> 2) >= kl) y = make_float4(pad, pad, pad, pad);
            } else {
                y.x = c < kl ? y.x : pad;
                y.y = c + 1 < kl ? y.y : pad;
                y.z = c + 2 < kl ? y.z : pad;
                y.w = c + 3 < kl ? y.w : pad;
            }
            v[it] = y;
        }
    };
    // statistics that cannot help are not taken, as in gemm_tile_chain
    int skip = 0, last_skip = 0;
    auto judge = [&](bool hopeless) {
        last_skip = hopeless ? min(2 * last_skip + 1, 15) : 0;
        skip = last_skip;
        return hopeless;
    };
    // registers -> LDS buffer, with the slice's flag fl and statistics (full: all of them)
    auto store_slice = [&](auto set, int k0, int fl, bool full) {
        constexpr int buf = decltype(set)::value;
        mend_op(va[buf], g.ta != 0, g.M - m0, g.K - k0, kPadA);
        mend_op(vb[buf], g.tb == 0, g.N - n0, g.K - k0, 0.0f);
        float* S = smem + buf * kFewBuf;
        auto put = [&](float* d, const float4 (&v)[2], bool kmaj) {
#pragma unroll
            for (int it = 0; it < 2; ++it) {
                const int f = tid + 256 * it;
                if (kmaj) {
                    float* q = d + 4 * (f & 3) * ROW + (f >> 2);
                    q[0] = v[it].x;
                    q[ROW] = v[it].y;
                    q[2 * ROW] = v[it].z;
                    q[3 * ROW] = v[it].w;
                } else {
                    *(float4*)(d + (f >> 5) * ROW + 4 * (f & 31)) = v[it];
                }
            }
        };
        put(S, va[buf], g.ta != 0);
        put(S + kFewB * ROW, vb[buf], g.tb == 0);
        if constexpr (kFlag) {
            float z = 0.0f;   // 0 * v summed: NaN as soon as one v is not finite
            auto sum = [&](const float4& v) {
                z = __builtin_fmaf(v.x, 0.0f, z);
                z = __builtin_fmaf(v.y, 0.0f, z);
                z = __builtin_fmaf(v.z, 0.0f, z);
                z = __builtin_fmaf(v.w, 0.0f, z);
            };
#pragma unroll
            for (int it = 0; it < 2; ++it) {
                sum(va[buf][it]);
                sum(vb[buf][it]);
            }
            if (z != 0.0f) flags[fl] = 1u;
        }
        if constexpr (kStat) {
            if (!full) {
                if constexpr (KIND == kChainMant10) {
                    uint32_t ma = 0u, mb = 0u, nb = ~0u;
                    auto top = [](uint32_t& m, const float4& v) {
                        m = max(max(m, __float_as_uint(v.x) << 1), __float_as_uint(v.y) << 1);
                        m = max(max(m, __float_as_uint(v.z) << 1), __float_as_uint(v.w) << 1);
                    };
                    auto low = [](uint32_t& m, const float4& v) {
                        m = min(min(m, (__float_as_uint(v.x) << 1) - 1u), (__float_as_uint(v.y) << 1) - 1u);
                        m = min(min(m, (__float_as_uint(v.z) << 1) - 1u), (__float_as_uint(v.w) << 1) - 1u);
                    };
#pragma unroll
                    for (int it = 0; it < 2; ++it) {
                        top(ma, va[buf][it]);
                        top(mb, vb[buf][it]);
                        low(nb, vb[buf][it]);
                    }
                    ma = wave_max_u32(ma);
                    mb = wave_max_u32(mb);
                    nb = wave_min_u32(nb) >> 24;
                    if (lane == 63)
                        *(uint4*)(stats + buf * 16 + wave * 4) = make_uint4(ma, 0u, mb, nb == 0u ? 1u : nb + 23u);
                }
                return;
            }
            SliceKey ka, kb;
#pragma unroll
            for (int it = 0; it < 2; ++it) {
                ka.add(va[buf][it]);
                kb.add(vb[buf][it]);
            }
            const uint4 w = make_uint4(wave_max_u32(ka.amax), wave_min_u32(ka.key),
                                       wave_max_u32(kb.amax), wave_min_u32(kb.key));
            if (lane == 63) *(uint4*)(stats + buf * 16 + wave * 4) = w;
        }
    };

    // the accumulator; binary16 and chunk 1: negated, from -0
    constexpr bool kNeg = KIND == kChainHalf || kStep;
    float acc = kNeg ? -0.0f : 0.0f;
    uint32_t h = 0x8000u;   // chunk 1, binary16: the accumulator while `held`
    bool held = KIND == kChainHalf && kStep;
    int accL = 1000;        // every accumulator of the wave is a multiple of 2^accL; -1000: unknown

    auto a_at = [&](const float* S, int k) { return *(const float4*)(S + row * ROW + k); };
    auto b_at = [&](const float* S, int k) { return *(const float4*)(S + (kFewB + colm) * ROW + k); };
    // use(a, b, st) for stages st < n (even) of four float4s of each operand, number j at k_of(st) + j
    // * dist: a stage is read while the one before computes, which hides the LDS latency of a lone
    // wave (8x4096x4096, binary16-shaped, e4m3 operands: 115 us with 4 k read ahead, 60 us so).
    auto stages = [&](const float* S, int n, int dist, auto k_of, auto use) {
        float4 a[2][4], b[2][4];
        auto fetch = [&](int set, int st) {
            const int k = k_of(st);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                a[set][j] = a_at(S, k + j * dist);
                b[set][j] = b_at(S, k + j * dist);
            }
        };
        fetch(0, 0);
        for (int st = 0; st < n; st += 2) {
            fetch(1, st + 1);
            __builtin_amdgcn_sched_barrier(0);
            use(a[0], b[0], st);
            __builtin_amdgcn_sched_barrier(0);
            fetch(0, st + 2 < n ? st + 2 : st);
            __builtin_amdgcn_sched_barrier(0);
            use(a[1], b[1], st + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // leaf(a, b) for every four k of [k0, k1), up to 31 more of the slice (past K they add -0)
    auto for_k4 = [&](const float* S, int k0, int k1, auto leaf) {
        stages(S, (k1 - k0 + 31) / 32 * 2, 4, [&](int st) { return k0 + 16 * st; },
               [&](const float4* a, const float4* b, int) {
#pragma unroll
                   for (int j = 0; j < 4; ++j) leaf(a[j], b[j]);
               });
    };
    auto directed = [&](const float* S, int k0, int k1) {
        // nothing computed from acc moves into the region; what else may is integer work and loads
        asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 2\n\ts_nop 1" : "+v"(acc));
        for_k4(S, k0, k1, [&](const float4& a, const float4& b) { few_fnma4_down<KIND>(a, b, acc, g); });
        asm volatile("s_nop 1\n\ts_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0\n\ts_nop 1" : "+v"(acc));
    };
    auto general = [&](const float* S, int k1) {
        const LeafGen L = leaf_gen(g);
        for (int k = 0; k < k1; ++k)
            acc = -(float)leaf_slow<LeafGen>((double)S[row * ROW + k] * (double)S[(kFewB + colm) * ROW + k],
                                             -(double)acc, L);
    };
    // the largest, least and lowest-bit figures of the wave's accumulators
    auto wave_hi = [&]() {
        return (uint32_t)__builtin_amdgcn_readlane((int)wave_max_u32(__float_as_uint(fabsf(acc))), 63);
    };
    auto wave_lsb = [&]() {
        const uint32_t x = __float_as_uint(acc);
        const uint32_t key = (((x << 1) - 1u) >> 24) + min((uint32_t)__builtin_ctz(x | 0x80000000u), 24u);
        return __builtin_amdgcn_readlane((int)wave_min_u32(key), 63) - 150;   // 129 for zeros
    };

    auto step_slice = [&](const float* S, int buf, int kmax, bool special, bool full) {
        if constexpr (KIND == kChainHalf) {
            // as gemm_tile_chain: one mixed FMA a k, redone if a result passed 65504
            if (!held && (!wave_in || __all((float)(_Float16)acc == acc && fabsf(acc) < 32768.0f))) {
                held = true;
                h = __builtin_bit_cast(uint16_t, (_Float16)acc);
            }
            if (held) {
                const uint32_t h0 = h;
                for_k4(S, 0, kmax, [&](const float4& a, const float4& b) { few_mix4(a, b, h); });
                if (wave_in && __any((h & 0x7C00u) == 0x7C00u)) {
                    acc = (float)__builtin_bit_cast(_Float16, (uint16_t)h0);
                    held = false;
                }
            }
            if (!held) general(S, kmax);
            return;
        }
        if (__builtin_expect(special, 0)) {
            general(S, kmax);
            accL = -1000;
            return;
        }
        if (!kStat || (KIND == kChainMant23 && !full)) {
            accL = -1000;
            directed(S, 0, kmax);
            return;
        }
        uint32_t amA = 0u, amB = 0u, kyA = ~0u, kyB = ~0u;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const uint4 v = *(const uint4*)(stats + buf * 16 + w * 4);
            amA = max(amA, v.x); kyA = min(kyA, v.y);
            amB = max(amB, v.z); kyB = min(kyB, v.w);
        }
        const int sL = !full ? -1000 : amA == 0u || amB == 0u ? 1000 : (int)kyA + (int)kyB - 300;
        const float pm = fmaxf(__uint_as_float(amA >> 1) * __uint_as_float(amB >> 1), 0x1p-126f) *
                         1.0000152587890625f;
        const bool hopeless = full && judge(__builtin_amdgcn_readfirstlane((int)(__float_as_uint(pm) >> 23)) - 126 >
                                            __builtin_amdgcn_readfirstlane(sL) + (KIND == kChainMant10 ? 39 : 24));
        // bounds for n leaves as gemm_tile_chain's for 32: every sum below 2^S, a multiple of 2^L
        if constexpr (KIND == kChainMant23) {
            for (int k = 0; k < kmax;) {
                const float hi = __uint_as_float(wave_hi());
                auto top = [&](float n) {
                    return (int)(__float_as_uint(__builtin_fmaf(n, pm, hi) * 1.0000152587890625f) >> 23) - 126;
                };
                const int S32 = top(33.0f);
                bool ok = S32 <= 127 && sL >= -149 && S32 <= sL + 24;
                if (ok && accL < sL) {
                    if (accL == -1000) accL = wave_lsb();
                    ok = accL >= -149 && S32 <= min(sL, accL) + 24;
                }
                if (!ok) {
                    accL = -1000;
                    const int k1 = hopeless ? kmax : min(k + 32, kmax);
                    directed(S, k, k1);
                    k = k1;
                    continue;
                }
                accL = min(accL, sL);
                const int S128 = top(129.0f), k1 = S128 <= 127 && S128 <= accL + 24 ? kmax : min(k + 32, kmax);
                for_k4(S, k, k1, [&](const float4& a, const float4& b) {
                    acc = __builtin_fmaf(-a.x, b.x, acc);
                    acc = __builtin_fmaf(-a.y, b.y, acc);
                    acc = __builtin_fmaf(-a.z, b.z, acc);
                    acc = __builtin_fmaf(-a.w, b.w, acc);
                });
                k = k1 == kmax ? kmax : k + 32;
            }
        } else if constexpr (KIND == kChainMant10) {
            const int bLsb = amB == 0u ? 1000 : (int)kyB - 150;
            const int bTop = amB == 0u ? -1000 : (int)(amB >> 24) - 127;
            const uint32_t hi = wave_hi();
            const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane(
                (int)wave_min_u32(__float_as_uint(fabsf(acc))), 63);
            // (1 + 2^-11)^128 = 1.06448...
            const float bnd = __builtin_fmaf(129.0f, pm, __uint_as_float(hi)) * 1.0646f;
            const int S2 = (int)(__float_as_uint(bnd) >> 23) - 126;
            const bool in = S2 <= 127;
            bool grid = in && sL >= -126 && S2 - sL <= 39;
            if (grid && accL == -1000) accL = wave_lsb();
            const int L = min(sL, accL);
            // the mixed FMA takes any FP32 b 2^hs, so B's bounds are the checked form's
            const int gLo = max(-24 - L, -126 - bLsb), gHi = min(min(15 - S2, 112), 126 - bTop);
            grid = grid && L >= -126 && gLo <= gHi;
            const int eLo = (int)(lo >> 23) - 127;
            const int cLo = max(-14 - eLo, -126 - bLsb);
            accL = grid ? L : -1000;
            if (grid || (in && lo != 0u && cLo <= gHi)) {
                const int hs = gHi;
                uint32_t u = __builtin_bit_cast(uint16_t, (_Float16)__builtin_ldexpf(acc, hs)), least = 0x7BFFu;
                auto scaled = [&](const float4& b) {
                    return make_float4(__builtin_ldexpf(b.x, hs), __builtin_ldexpf(b.y, hs),
                                       __builtin_ldexpf(b.z, hs), __builtin_ldexpf(b.w, hs));
                };
                if (grid)
                    for_k4(S, 0, kmax, [&](const float4& a, const float4& b) { few_mix4(a, scaled(b), u); });
                else
                    for_k4(S, 0, kmax, [&](const float4& a, const float4& b) { few_mix4_least(a, scaled(b), u, least); });
                if (grid || __all((least & 0xFFFFu) > 0x0400u)) {   // 2^-14
                    acc = __builtin_ldexpf((float)__builtin_bit_cast(_Float16, (uint16_t)u), -hs);
                    return;
                }
            }
            directed(S, 0, kmax);
        }
    };
    auto chunk_slice = [&](const float* S, int kmax, bool special) {
        float p[4], top = 0.0f;
        const float acc0 = acc;
        auto leaves = [&]() {
            if constexpr (KIND == kChainHalf) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    acc = mix_sub16(acc, p[j]);
                    top = fmaxf(top, fabsf(acc));
                }
            } else {
                if constexpr (KIND == kChainMant)
                    if (special) {   // wave-uniform: a NaN sum to the one quiet pattern
#pragma unroll
                        for (int j = 0; j < 4; ++j) p[j] = p[j] != p[j] ? __uint_as_float(0x7FC00000u) : p[j];
                    }
                few_add4<KIND>(p, acc, g);
            }
        };
        // four chunks' sums side by side; a chunk past K sums to 0, which changes nothing
        constexpr int PER = CHUNK <= 4 ? 1 : CHUNK / 4;   // stages per four chunks
        constexpr int KST = CHUNK <= 4 ? 32 : CHUNK == 8 ? 32 : 4 * CHUNK;   // k of an even number of stages
        stages(S, (kmax + KST - 1) / KST * (KST / 16), CHUNK <= 4 ? 4 : CHUNK,
               [&](int st) { return CHUNK <= 4 ? 16 * st : st / PER * 4 * CHUNK + st % PER * 4; },
               [&](const float4* a, const float4* b, int st) {
                   if constexpr (CHUNK == 2) {
#pragma unroll
                       for (int i = 0; i < 4; i += 2) {
#pragma unroll
                           for (int j = 0; j < 2; ++j) {
                               const float4 &x = a[i + j], &y = b[i + j];
                               p[2 * j] = __builtin_fmaf(x.y, y.y, __builtin_fmaf(x.x, y.x, 0.0f));
                               p[2 * j + 1] = __builtin_fmaf(x.w, y.w, __builtin_fmaf(x.z, y.z, 0.0f));
                           }
                           leaves();
                       }
                       return;
                   }
                   const bool first = PER == 1 || st % PER == 0;
#pragma unroll
                   for (int j = 0; j < 4; ++j) {
                       p[j] = __builtin_fmaf(a[j].x, b[j].x, first ? 0.0f : p[j]);
                       p[j] = __builtin_fmaf(a[j].y, b[j].y, p[j]);
                       p[j] = __builtin_fmaf(a[j].z, b[j].z, p[j]);
                       p[j] = __builtin_fmaf(a[j].w, b[j].w, p[j]);
                   }
                   if (PER == 1 || st % PER == PER - 1) leaves();
               });
        if constexpr (KIND == kChainHalf)
            if (__builtin_expect(wave_in && __any(top >= g.half_top), 0)) {   // the top binade: the slice again
                acc = acc0;
                for (int k = 0; k < kmax; k += CHUNK) {
                    float x = 0.0f;
                    for (int i = 0; i < CHUNK; ++i)
                        x = __builtin_fmaf(S[row * ROW + k + i], S[(kFewB + colm) * ROW + k + i], x);
                    float t = mix_sub16(acc, x);
                    if (fabsf(t) >= g.half_top) t = chain_half_slow(x, acc, leaf_gen(g));
                    acc = t;
                }
            }
    };

    // Flags three in turn as in gemm_tile_chain: slice s reads flag s % 3 between its barrier and
    // the next, the store of slice s + 1 sets the next one, the one after is cleared.
    if constexpr (kFlag) {
        if (tid < 3) flags[tid] = 0u;
        lds_barrier();
    }
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    int fs = 0;
    bool full = true;   // the statistics of the slice in LDS
    auto slice = [&](auto cur, auto nxt, int k0) {   // slice k0 is in buffer `cur`
        lds_barrier();
        const int fn = fs == 2 ? 0 : fs + 1;
        bool special = false;
        if constexpr (kFlag) {
            special = __builtin_amdgcn_readfirstlane((int)flags[fs]) != 0;
            if (tid == 0) flags[fn == 2 ? 0 : fn + 1] = 0u;
        }
        load_slice(cur, k0 + 2 * BK);
        const float* S = smem + cur.value * kFewBuf;
        const int kmax = min(BK, g.K - k0);
        if constexpr (kStep) step_slice(S, cur.value, kmax, special, full);
        else chunk_slice(S, kmax, special);
        if (k0 + BK < g.K) {
            full = skip == 0;
            skip = full ? 0 : skip - 1;
            store_slice(nxt, k0 + BK, fn, full);
        }
        fs = fn;
    };
    if (g.K > 0) {
        load_slice(P0{}, 0);
        load_slice(P1{}, BK);
        store_slice(P0{}, 0, 0, true);
    }
    for (int k0 = 0; k0 < g.K; k0 += 2 * BK) {
        slice(P0{}, P1{}, k0);
        if (k0 + BK < g.K) slice(P1{}, P0{}, k0 + BK);
    }
    if (KIND == kChainHalf && kStep && held) acc = (float)__builtin_bit_cast(_Float16, (uint16_t)h);

    const int gm = m0 + row, gn = n0 + colm;
    if (gm >= g.M || gn >= g.N) return;
    const float a = kNeg ? -acc : acc;
    float d = g.alpha * a;
    if (g.beta != 0.0f) d = __builtin_fmaf(g.alpha, a, g.beta * gld(g.C + (int64_t)gm * g.ldc + gn));
    gst(g.D + (int64_t)gm * g.ldd + gn, d);
}

}  // namespace lofamd
