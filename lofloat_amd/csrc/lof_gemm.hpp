// lof_gemm.hpp -- host-side interface of the GEMM launcher, shared with the grouped path.
#pragma once

#include <hip/hip_runtime.h>

#include "lof_gemm_kernels.hpp"
#include "lof_gemm_mfma.hpp"
#include "lofloat.h"

namespace lofamd {

lof_status prepare_gemm(const lof_gemm_desc* d, GemmArgs* g);
void set_fast_path(GemmArgs* g, bool on, int m);
// Whether the chunk-sum kernels take this product (g->chain); `conv`: B is gathered, not read
// through ldb.  prepare_gemm calls it for a stored B.
void set_chain(GemmArgs* g, bool conv);
// Tile of the chunk-sum kernels for an M x N product, and its launch.  few: the 16x16 tile takes it;
// directed: a mantissa-only accumulator at chunk 1, 10 and 23 bits aside; half: a binary16-shaped one.
int chain_default_tile(int64_t M, int64_t N, int chunk, bool few, bool directed, bool half);
lof_status launch_chain(const GemmArgs& g, int tile, hipStream_t st, const char* what);
lof_status launch_gemm(const GemmArgs& g, int config, hipStream_t st);
int gemm_default_config(const GemmArgs& g);   // the untuned config of lof_gemm_f32
int gemm_num_configs();
int gemm_config_bm(int c);
int gemm_config_bn(int c);
// the chunk lengths whose sums can run on MFMA (2, 4, 8, 16, 32)
bool gemm_chunk_fits_mfma(int chunk);

}  // namespace lofamd
