// lof_gemm_chain_mant10.hip -- chunk-1 GEMM kernels, accumulator: mantissa-only, 10 bits.
#include "lof_gemm_chain_table.hpp"

namespace lofamd {
extern const ChainTable kChainTableMant10 = LOF_CHAIN_TABLE1(kChainMant10);
}  // namespace lofamd
