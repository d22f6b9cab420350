// lof_gemm_chain_mant23.hip -- chunk-sum GEMM kernels, accumulator: mantissa-only, 23 bits.
#include "lof_gemm_chain_table.hpp"

namespace lofamd {
extern const ChainTable kChainTableMant23 = LOF_CHAIN_TABLE(kChainMant23);
}  // namespace lofamd
