// mttkrp_x3_w8.hip -- the 8-wave instances of the fp32 MTTKRP, with the ALS job.
#include "mttkrp_x3.hpp"
#include "mttkrp_x3_kernel.hpp"

namespace tenrso {

const void* mttkrp_x3_kernel_w8(int nt, bool case_b, bool wv, int xl) {
  if (nt == 1) return x3_pick<1, 8, 1>(case_b, wv, xl);
  if (nt == 2) return x3_pick<2, 8, 1>(case_b, wv, xl);
  return x3_pick<4, 8, 1>(case_b, wv, xl);
}

}  // namespace tenrso
