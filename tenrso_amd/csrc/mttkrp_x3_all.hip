// mttkrp_x3_all.hip -- the fp32 MTTKRP kernel over all modes of a tensor.
//
// A launch a mode leaves the GPU idle between the last workgroups of one and the first
// data of the next; here a CU goes on with the next mode's workgroups.  With whole
// windows the block loads are left to the compiler here (x3_tile's OPAQUE): other
// workgroups cover their start, and X streams better for it (X from memory each time: 96^4
// rank 32 199 us against 207, 512x512x128 rank 32 64 against 69; with masked windows
// 250^3 rank 16 takes 49 that way, 43 this).
#include "mttkrp_x3.hpp"
#include "mttkrp_x3_kernel.hpp"

namespace tenrso {

namespace {

template <int NT, bool WV, int XLA, int XLB>
__global__ __launch_bounds__(256) void mttkrp_x3_all(const float* __restrict__ X, AllModesArgs p) {
  constexpr int WAVES = 4;
  __shared__ __attribute__((aligned(16))) float smem[x3_lds<NT, WAVES>() / 4];
  __shared__ float wmin[WAVES];
  __shared__ int redo;
  int m = 0;
  while (m + 1 < p.nd && blockIdx.x >= p.first[m + 1]) ++m;
  const int tile = (int)(blockIdx.x - p.first[m]);
  const KernArgs a = p.a[m];
  if (m == p.nd - 1) x3_tile<NT, WAVES, true, WV, XLB, false, XLB != 0>(X, a, p.partial[m], tile, smem, wmin, redo);
  else x3_tile<NT, WAVES, false, WV, XLA, false, XLA != 0>(X, a, p.partial[m], tile, smem, wmin, redo);
}

template <int NT, bool WV>
const void* pick(int xla, int xlb) {
  if (xla == 0)
    return xlb == 0 ? reinterpret_cast<const void*>(mttkrp_x3_all<NT, WV, 0, 0>)
                    : reinterpret_cast<const void*>(mttkrp_x3_all<NT, WV, 0, 1>);
  return xlb == 0 ? reinterpret_cast<const void*>(mttkrp_x3_all<NT, WV, 1, 0>)
                  : reinterpret_cast<const void*>(mttkrp_x3_all<NT, WV, 1, 1>);
}

}  // namespace

const void* mttkrp_x3_kernel_all(int nt, bool wv, int xla, int xlb) {
  if (nt == 1) return wv ? pick<1, true>(xla, xlb) : pick<1, false>(xla, xlb);
  if (nt == 2) return wv ? pick<2, true>(xla, xlb) : pick<2, false>(xla, xlb);
  return wv ? pick<4, true>(xla, xlb) : pick<4, false>(xla, xlb);
}

}  // namespace tenrso
