// contract_block_kernel for complex128, nz = 32 to 47.
#include "contract_block.h"

namespace xtr {

bool contract_block_c128_d(const ApplyArgs &a, hipStream_t s) { return contract_block_range<double, 32, 47>(a, s); }

}  // namespace xtr
