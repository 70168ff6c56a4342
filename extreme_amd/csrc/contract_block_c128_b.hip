// contract_block_kernel for complex128, nz = 13 to 20.
#include "contract_block.h"

namespace xtr {

bool contract_block_c128_b(const ApplyArgs &a, hipStream_t s) { return contract_block_range<double, 13, 20>(a, s); }

}  // namespace xtr
