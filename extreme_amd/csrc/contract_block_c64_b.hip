// contract_block_kernel for complex64, nz = 17 to 31.
#include "contract_block.h"

namespace xtr {

bool contract_block_c64_b(const ApplyArgs &a, hipStream_t s) { return contract_block_range<float, 17, 31>(a, s); }

}  // namespace xtr
