// lof_gemm_chain_mant.hip -- chunk-sum GEMM kernels, accumulator: mantissa-only, 1 to 22 bits.
#include "lof_gemm_chain_table.hpp"

namespace lofamd {
extern const ChainTable kChainTableMant = LOF_CHAIN_TABLE(kChainMant);
}  // namespace lofamd
