// contract_block_kernel for complex128, nz = 21 to 31.
#include "contract_block.h"

namespace xtr {

bool contract_block_c128_c(const ApplyArgs &a, hipStream_t s) { return contract_block_range<double, 21, 31>(a, s); }

}  // namespace xtr
