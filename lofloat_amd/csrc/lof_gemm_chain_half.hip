// lof_gemm_chain_half.hip -- chunk-sum GEMM kernels, accumulator: binary16-shaped.
#include "lof_gemm_chain_table.hpp"

namespace lofamd {
extern const ChainTable kChainTableHalf = LOF_CHAIN_TABLE(kChainHalf);
}  // namespace lofamd
