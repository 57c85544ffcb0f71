// mttkrp_x3_n8.hip -- the fp32 MTTKRP instances of 65 to 128 ranks, with the
// wide-rank ALS job.
#include "mttkrp_x3.hpp"
#include "mttkrp_x3_kernel.hpp"

namespace tenrso {

const void* mttkrp_x3_kernel_n8(bool case_b, bool wv, int xl) { return x3_pick<8, 8, 2>(case_b, wv, xl); }

}  // namespace tenrso
