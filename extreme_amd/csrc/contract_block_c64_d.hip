// contract_block_kernel for complex64, nz = 48 to 63.
#include "contract_block.h"

namespace xtr {

bool contract_block_c64_d(const ApplyArgs &a, hipStream_t s) { return contract_block_range<float, 48, 63>(a, s); }

}  // namespace xtr
