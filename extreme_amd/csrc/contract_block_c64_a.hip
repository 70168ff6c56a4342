// contract_block_kernel for complex64, nz = 1 to 16.
#include "contract_block.h"

namespace xtr {

bool contract_block_c64_a(const ApplyArgs &a, hipStream_t s) { return contract_block_range<float, 1, 16>(a, s); }

}  // namespace xtr
