// contract_block_kernel for complex64, nz = 32 to 47.
#include "contract_block.h"

namespace xtr {

bool contract_block_c64_c(const ApplyArgs &a, hipStream_t s) { return contract_block_range<float, 32, 47>(a, s); }

}  // namespace xtr
