// mttkrp_x3.hpp -- the fp32 MTTKRP kernels on the bf16 matrix cores
// (mttkrp_x3_kernel.hpp).
#pragma once

namespace tenrso {

// The instance for nt rank tiles of 16 (1, 2 or 4), case A (q-contiguous) or B, wv
// (16-byte window loads) and the load form xl (0, 1, or 4 in case A), to be
// launched with (const float* X, KernArgs, float* partial, AlsJob, int has_job):
// 8 waves, able to run the ALS job as workgroup 0, or 4 waves without it.
const void* mttkrp_x3_kernel_w8(int nt, bool case_b, bool wv, int xl);
const void* mttkrp_x3_kernel_w4(int nt, bool case_b, bool wv, int xl);
// The 4-wave instances that also leave the sum of squares of X (KernArgs::norm).
const void* mttkrp_x3_kernel_norm(int nt, bool case_b, bool wv, int xl);
// Eight rank tiles, 8 waves, able to run the wide-rank job.
const void* mttkrp_x3_kernel_n8(bool case_b, bool wv, int xl);

// All modes in one launch (AllModesArgs); xla: the load form of modes 0 .. nd-2, xlb:
// of the last.  4 waves a workgroup.
const void* mttkrp_x3_kernel_all(int nt, bool wv, int xla, int xlb);

}  // namespace tenrso
