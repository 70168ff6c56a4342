// contract_block_kernel for complex128, nz = 1 to 12.
#include "contract_block.h"

namespace xtr {

bool contract_block_c128_a(const ApplyArgs &a, hipStream_t s) { return contract_block_range<double, 1, 12>(a, s); }

}  // namespace xtr
