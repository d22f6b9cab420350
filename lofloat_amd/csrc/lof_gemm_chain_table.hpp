// lof_gemm_chain_table.hpp -- the chunk-sum kernels of one accumulator kind: a table over tiles
// and chunks, instantiated by one source file per kind (they compile side by side).
#pragma once

#include "lof_gemm_chain.hpp"
#include "lof_gemm_few.hpp"

namespace lofamd {

// Tile t of the tables below:
//   0, 1   128x128 and 64x64: blocks of 32x32, slices of 32 k.  (128x64 and 64x128, two blocks a
//          wave, are slower than both at 4096^3 and at 1537 x 3001 x 2047 on every kind.)
//   2      32x32: four 16x16 blocks, slices of 64 k
//   3, 4   16x64 and 64x16: slices of 128 k
//   5      16x16, an output a lane (lof_gemm_few.hpp)
// The short blocks need few outputs for a full chip, and longer slices per barrier because a
// slice of one block is only a quarter as long on the matrix cores.
using ChainT0 = ChainTile<32, 2, 2, 2, 2, 32>;
using ChainT1 = ChainTile<32, 2, 2, 1, 1, 32>;
using ChainT2 = ChainTile<16, 2, 2, 1, 1, 64>;
using ChainT3 = ChainTile<16, 1, 4, 1, 1, 128>;
using ChainT4 = ChainTile<16, 4, 1, 1, 1, 128>;
constexpr int kChainTiles = 6;

// Tile t of `tiles` in launch order: each XCD (workgroups go to the 8 XCDs in turn) takes a
// contiguous run of tiles, walked in groups of 8 tile rows, so that the tiles in flight on one
// XCD share their A and B slices in its L2.
__device__ __forceinline__ int2 chain_tile_of(unsigned id, unsigned tm, unsigned tn) {
    const unsigned total = tm * tn, q = total >> 3, r = total & 7u, x = id & 7u;
    const unsigned t = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + (id >> 3);
    const unsigned grp = t / (8u * tn), in = t - grp * 8u * tn, rows = min(8u, tm - grp * 8u);
    return make_int2((int)(grp * 8u + in % rows), (int)(in / rows));
}

// Waves per SIMD the registers are held to: 2 for 32 or more sums a wave, 4 else.
template <class T>
constexpr int kChainWaves = T::WMB * T::WNB * T::NR >= 32 ? 2 : 4;

template <class T, int CHUNK, int KIND, bool CONV>
__global__ __launch_bounds__(256, kChainWaves<T>) void k_gemm_chain(GemmArgs g, unsigned tm,
                                                                    unsigned tn) {
    __shared__ __align__(16) float smem[T::SMEM_FLOATS];
    const int2 t = chain_tile_of(blockIdx.x, tm, tn);
    // Co-resident workgroups (ids 256 apart share a CU) get different priorities, so that one is
    // between its MFMA runs while another is inside one (4096^3, 64x64: 1.411 -> 1.353 ms).
    switch ((blockIdx.x >> 8) & 3u) {
    case 1: __builtin_amdgcn_s_setprio(1); break;
    case 2: __builtin_amdgcn_s_setprio(2); break;
    case 3: __builtin_amdgcn_s_setprio(3); break;
    default: break;
    }
    gemm_tile_chain<T, CHUNK, KIND, CONV>(g, t.x, t.y, (int)threadIdx.x, smem);
}

template <int CHUNK, int KIND>
__global__ __launch_bounds__(256, 4) void k_gemm_few(GemmArgs g, unsigned tm, unsigned tn) {
    __shared__ __align__(16) float smem[kFewSmem];
    const int2 t = chain_tile_of(blockIdx.x, tm, tn);
    gemm_tile_few<CHUNK, KIND>(g, t.x, t.y, (int)threadIdx.x, smem);
}

using ChainKernel = void (*)(GemmArgs, unsigned, unsigned);

// [tile][log2(chunk)]; nullptr where a chunk of 2 is shorter than the block's MFMA, and for chunk
// 1 on the widest tile
struct ChainTable {
    ChainKernel gemm[kChainTiles][6];
    ChainKernel conv[kChainTiles][6];
};

template <class T, int CHUNK, int KIND, bool CONV>
constexpr ChainKernel chain_kernel() {
    if constexpr (CHUNK == 1 ? T::WMB == 1 : CHUNK >= T::KI) return k_gemm_chain<T, CHUNK, KIND, CONV>;
    else return nullptr;
}

#define LOF_CHAIN_ROW(T, KIND, CONV)                                                        \
    {chain_kernel<T, 1, KIND, CONV>(), chain_kernel<T, 2, KIND, CONV>(),                     \
     chain_kernel<T, 4, KIND, CONV>(), chain_kernel<T, 8, KIND, CONV>(),                     \
     chain_kernel<T, 16, KIND, CONV>(), chain_kernel<T, 32, KIND, CONV>()}
// the convolution gathers its B slice, which costs the wide tiles more than it gives
#define LOF_CHAIN_TABLE(KIND)                                                               \
    {{LOF_CHAIN_ROW(ChainT0, KIND, false), LOF_CHAIN_ROW(ChainT1, KIND, false),              \
      LOF_CHAIN_ROW(ChainT2, KIND, false), LOF_CHAIN_ROW(ChainT3, KIND, false),              \
      LOF_CHAIN_ROW(ChainT4, KIND, false),                                                   \
      {k_gemm_few<1, KIND>, k_gemm_few<2, KIND>, k_gemm_few<4, KIND>, k_gemm_few<8, KIND>,   \
       k_gemm_few<16, KIND>, k_gemm_few<32, KIND>}},                                         \
     {{}, LOF_CHAIN_ROW(ChainT1, KIND, true), LOF_CHAIN_ROW(ChainT2, KIND, true),            \
      LOF_CHAIN_ROW(ChainT3, KIND, true), {}, {}}}

// chunk 1 alone (longer chunks of a 10-bit accumulator are kChainMant's)
#define LOF_CHAIN_ROW1(T, KIND, CONV) {chain_kernel<T, 1, KIND, CONV>(), {}, {}, {}, {}, {}}
#define LOF_CHAIN_TABLE1(KIND)                                                              \
    {{{}, LOF_CHAIN_ROW1(ChainT1, KIND, false), LOF_CHAIN_ROW1(ChainT2, KIND, false),        \
      LOF_CHAIN_ROW1(ChainT3, KIND, false), LOF_CHAIN_ROW1(ChainT4, KIND, false),            \
      {k_gemm_few<1, KIND>, {}, {}, {}, {}, {}}},                                            \
     {{}, LOF_CHAIN_ROW1(ChainT1, KIND, true), LOF_CHAIN_ROW1(ChainT2, KIND, true),          \
      LOF_CHAIN_ROW1(ChainT3, KIND, true), {}, {}}}

extern const ChainTable kChainTableMant, kChainTableMant10, kChainTableMant23, kChainTableHalf;

// Leading dimensions past those of the tiles, 16x16 aside, which takes any (`conv`: B is gathered).
inline bool chain_rows_far_apart(const GemmArgs& g, bool conv) {
    return g.lda > kChainMaxLd || (!conv && g.ldb > kChainMaxLd);
}

// The dimensions of tile t.
struct ChainDims { int bm, bn; };
constexpr ChainDims kChainDims[kChainTiles] = {{128, 128}, {64, 64}, {32, 32}, {16, 64}, {64, 16}, {16, 16}};
// Workgroups of one launch: HIP takes fewer than 2^32 threads in a dimension of the grid.
constexpr int64_t kChainMaxTiles = (1 << 24) - 1;
inline int64_t chain_tiles(int64_t M, int64_t N, int t) {
    return ((M + kChainDims[t].bm - 1) / kChainDims[t].bm) * ((N + kChainDims[t].bn - 1) / kChainDims[t].bn);
}
// GEMM configs 5.. (lof_gemm.hip) and the tile each runs on here (-1: 128x64 and 64x128, not here), and back
constexpr int kChainTileOf[8] = {0, -1, 1, -1, 2, 3, 4, 5};
constexpr int kChainConfigOf[kChainTiles] = {5, 7, 9, 10, 11, 12};

}  // namespace lofamd
