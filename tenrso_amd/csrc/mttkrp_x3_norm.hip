// mttkrp_x3_norm.hip -- the 4-wave instances of the fp32 MTTKRP that also sum the
// squares of X.
#include "mttkrp_x3.hpp"
#include "mttkrp_x3_kernel.hpp"

namespace tenrso {

const void* mttkrp_x3_kernel_norm(int nt, bool case_b, bool wv, int xl) {
  if (nt == 1) return x3_pick<1, 4, 0, true>(case_b, wv, xl);
  if (nt == 2) return x3_pick<2, 4, 0, true>(case_b, wv, xl);
  return x3_pick<4, 4, 0, true>(case_b, wv, xl);
}

}  // namespace tenrso
