// cp_init.hip -- the SVD-based CP initialisations (InitStrategy::Svd, Nnsvd,
// LeverageScore of tenrso-decomp cp/helpers.rs:232-373) on the device.
//
// Per mode k (X viewed as [P, I, Q], I = I_k, J = P*Q columns of the unfolding):
//   1. K = X_(k) X_(k)^T (I x I, FP64): the left singular vectors of X_(k) are the
//      eigenvectors of K and its singular values the square roots of K's
//      eigenvalues.  Split-K tiles on the FP64 matrix cores, then a reduction that
//      also mirrors the upper triangle.
//   2. Two-sided block Jacobi, every mode at once: pairs of 32-wide blocks (circle
//      method) are diagonalised by one workgroup each, their 64 x 64 rotations
//      applied to K and to the eigenvectors by 64 x 64 tiles over the whole GPU,
//      until the off-diagonal mass is below 1e-14 of the diagonal; then the top R
//      eigenpairs in descending order.  The sign of each eigenvector is fixed so
//      that its entry of largest magnitude is positive (an SVD's signs are
//      arbitrary; the third-party SVD behind the reference does not document one).
//   3. Nnsvd only: ||max(v_r, 0)|| and ||max(-v_r, 0)|| of the right singular
//      vectors v_r = X_(k)^T u_r / s_r, streamed over the columns of X_(k).
//   4. The factor: Svd u_r; LeverageScore u_r sqrt(s_r) sqrt(l_i I) with the
//      normalised leverage scores l_i; Nnsvd the larger-product sign part of u_r
//      scaled by sqrt(s_r * prod) (helpers.rs:265-310).  Columns past
//      min(R, I, J) come from the caller's N(0, 0.01) draws (|.| for Nnsvd,
//      times l_i for LeverageScore), as in the reference.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <random>
#include <vector>

#include "common.hpp"
#include "cp_init.hpp"
#include "mttkrp.hpp"

namespace tenrso {

constexpr int EIG_NMAX = 1024;  // bound of the mode sizes
constexpr int INIT_RMAX = 128;  // rank bound of the SVD-based initialisations (that of the ALS)
// Sweeps queued before the host first looks whether every mode has converged (it takes
// 11 to 19 at 256 to 1024 rows), and the bound.
constexpr int JACOBI_FIRST = 12, JACOBI_SWEEPS = 60;
constexpr double JACOBI_TOL = 1e-14;       // off-diagonal over diagonal, Frobenius norms
// An entry over sqrt(w_i w_j), the weights of its row and column: rounding noise up to
// the first (2^-46 to 2^-50 give the same vectors in 13 to 17 sweeps at 256 rows); none
// above the second once done, so that small rows beside large ones converge as well.
constexpr double JACOBI_NOISE = 0x1p-47, JACOBI_ROW = 0x1p-34;

namespace {

typedef double doublex4 __attribute__((ext_vector_type(4)));

constexpr int GT = 64;  // Gram tile
constexpr int GK = 32;  // columns staged per step

// Gram partials: workgroup (tile pair, split) sums the columns [j0, j1) of its split
// for a 64 x 64 tile (ti <= tj) of K on the FP64 matrix cores; each of its 4 waves
// owns 32 x 32 of it.  32 columns of both row tiles at a time go through LDS as fp32
// (the next ones loaded meanwhile); element (i, j) of the unfolding is X[p, i, q]
// with (p, q) = (j / Q, j % Q).  Bound: the FP64 matrix cores, 74 us at 256 rows of
// 65536 columns at 73 TFLOP/s (32 x 32 tiles of VALU FMAs took 526 us).
__global__ __launch_bounds__(256) void unfold_gram_partial_kernel(const float* __restrict__ X, i64 P, i64 I, i64 Q,
                                                                  int nt, int splits, double* __restrict__ part) {
  __shared__ float sA[GT][GK + 4], sB[GT][GK + 4];
  int t = blockIdx.x, ti = 0;
  while (t >= nt - ti) {
    t -= nt - ti;
    ++ti;
  }
  const int tj = ti + t;
  const int split = blockIdx.y;
  const i64 J = P * Q;
  const i64 j0 = J * split / splits, j1 = J * (split + 1) / splits;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, q4 = lane >> 4, l16 = lane & 15;
  constexpr int PER = GT * GK / 256;
  // a thread stages one column of a step: rows tid / 32 + 8 e, or (Q == 1, where
  // consecutive rows are contiguous) one row: columns tid / 64 + 4 e
  const bool rowwise = Q != 1;
  float ra[PER], rb[PER];
  auto load = [&](i64 jb) {
    if (rowwise) {
      const i64 j = jb + (tid & 31);
      const bool ok = j < j1;
      const i64 p = ok ? ((J >> 32) ? j / Q : (i64)((uint32_t)j / (uint32_t)Q)) : 0;
      const float* x = X + (ok ? p * I * Q + (j - p * Q) : 0);
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        const i64 ia = (i64)ti * GT + (tid >> 5) + 8 * e, ib = (i64)tj * GT + (tid >> 5) + 8 * e;
        ra[e] = ok && ia < I ? x[ia * Q] : 0.f;
        rb[e] = ok && ib < I ? x[ib * Q] : 0.f;
      }
    } else {
      const i64 ia = (i64)ti * GT + lane, ib = (i64)tj * GT + lane;
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        const i64 j = jb + wave + 4 * e;
        ra[e] = j < j1 && ia < I ? X[j * I + ia] : 0.f;
        rb[e] = j < j1 && ib < I ? X[j * I + ib] : 0.f;
      }
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int r = rowwise ? (tid >> 5) + 8 * e : lane, c = rowwise ? (tid & 31) : wave + 4 * e;
      sA[r][c] = ra[e];
      sB[r][c] = rb[e];
    }
  };
  doublex4 acc[2][2];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < 2; ++v) acc[u][v] = doublex4{0.0, 0.0, 0.0, 0.0};
  const int ar = 32 * (wave >> 1) + l16, br = 32 * (wave & 1) + l16;
  load(j0);
  for (i64 jb = j0; jb < j1; jb += GK) {
    store();
    __syncthreads();
    if (jb + GK < j1) load(jb + GK);
#pragma unroll
    for (int kk = 0; kk < GK / 4; ++kk) {
      double av[2], bv[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        av[u] = (double)sA[ar + 16 * u][4 * kk + q4];
        bv[u] = (double)sB[br + 16 * u][4 * kk + q4];
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v) acc[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[u], bv[v], acc[u][v], 0, 0, 0);
    }
    __syncthreads();
  }
  double* out = part + (i64)split * I * I;
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const i64 i = (i64)ti * GT + 32 * (wave >> 1) + 16 * u + 4 * e + q4;
        const i64 i2 = (i64)tj * GT + 32 * (wave & 1) + 16 * v + l16;
        if (i < I && i2 < I) out[i * I + i2] = acc[u][v][e];
      }
}

// The eigenproblem of every mode (by value to the kernels below).  n is padded to a
// multiple N of 64 with zero rows and columns, which no rotation touches.
struct EigMode {
  double* A;    // N x N: K, then diagonal
  double* V;    // N x N: eigenvectors in columns
  double* Q;    // [N / 64][64][64]: the rotations of a round
  int* done;
  double* w;    // N: weights of the rows (noise_root)
  double* U;    // n x R: eigenvectors of the top R, descending
  double* lam;  // R
  int n, N;
};
struct EigArgs {
  EigMode m[MAXD];
  int R;
};

// K[i][i2] = sum of the split partials, for tile(i) <= tile(i2), mirrored below; V = 1
__global__ __launch_bounds__(256) void unfold_gram_reduce_kernel(const double* __restrict__ part, int splits,
                                                                 EigMode m) {
  const i64 e = (i64)blockIdx.x * 256 + threadIdx.x, I = m.n, N = m.N;
  if (e == 0) *m.done = 0;
  if (e >= N * N) return;
  const i64 i = e / N, i2 = e - (e / N) * N;
  m.V[e] = i == i2 ? 1.0 : 0.0;
  if (i >= I || i2 >= I) {
    m.A[e] = 0.0;
    if (i == i2) m.w[i] = 0.0;
    return;
  }
  if (i / GT > i2 / GT) return;
  double s = 0.0;
  for (int k = 0; k < splits; ++k) s += part[(i64)k * I * I + i * I + i2];
  m.A[i * N + i2] = s;
  m.A[i2 * N + i] = s;
  if (i == i2) m.w[i] = s;
}

// pair k of round r of the circle method over `count` (even) indices
__device__ __forceinline__ void circle_pair(int count, int r, int k, int& a, int& b) {
  a = k == 0 ? r : (r + k) % (count - 1);
  b = k == 0 ? count - 1 : (r - k + (count - 1)) % (count - 1);
}

// 1 / sqrt(x), two Newton steps
__device__ __forceinline__ double rsqrt_newton(double x) {
  double y = __builtin_amdgcn_rsq(x);
#pragma unroll
  for (int k = 0; k < 2; ++k) y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
  return y;
}

// The Jacobi rotation (c, s) of a = a_qq - a_pp and b = 2 a_pq != 0:
// t = b / (a + sign(a) sqrt(a^2 + b^2)), c = 1 / sqrt(1 + t^2), s = t c.  By
// approximate reciprocals refined to full precision, a third of the chain of two
// divisions and two square roots; those where a^2 + b^2 leaves the exponent range.
__device__ __forceinline__ void rotation(double a, double b, double& c, double& s) {
  const double h2 = fma(a, a, b * b);
  double t;
  if (h2 > 0x1p-900 && h2 < 0x1p900) {
    const double den = fma(h2, rsqrt_newton(h2), fabs(a));
    double r = __builtin_amdgcn_rcp(den);
    r = fma(r, fma(-den, r, 1.0), r);
    r = fma(r, fma(-den, r, 1.0), r);
    t = (a >= 0.0 ? b : -b) * r;
    c = rsqrt_newton(fma(t, t, 1.0));
  } else {
    const double th = a / b;
    t = (th >= 0.0 ? 1.0 : -1.0) / (fabs(th) + sqrt(fma(th, th, 1.0)));
    c = 1.0 / sqrt(fma(t, t, 1.0));
  }
  s = t * c;
}

template <int THREADS>
__device__ __forceinline__ double block_sum(double v, double* red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < THREADS / 64; ++w) s += red[w];
  __syncthreads();
  return s;
}

// Rounding noise: an entry up to r_i r_j.  K_ij was summed with an error relative to
// sqrt(K_ii K_jj), so the weights start as the diagonal of K and are carried through the
// rotations as variances are.  (Relative to the whole matrix instead, rows of a small
// scale come out as they went in: slices of 1e-6 beside ordinary ones.)
__device__ __forceinline__ double noise_root(double w) { return sqrt(JACOBI_NOISE * w); }

// done once the off-diagonal mass is below JACOBI_TOL of the diagonal's; one workgroup a
// mode.  Entries that are rounding errors count as zero and are not rotated: in the null
// space of an exact low-rank tensor there is nothing else, diagonal entries included, so
// every rotation there is one of about 45 degrees, and the block method then converges
// linearly.  (256 rows, rank 64, weights down to 1e-4: 17 sweeps; with those rotations
// 1e-10 off after 24, and vectors off by 7e-6 after 18.)
__global__ __launch_bounds__(1024) void jacobi_check_kernel(EigArgs a) {
  __shared__ double red[16], rt[EIG_NMAX];
  const EigMode& m = a.m[blockIdx.x];
  if (*m.done) return;
  const i64 N = m.N;
  double off = 0.0, dia = 0.0, large = 0.0;
  for (i64 i = threadIdx.x; i < N; i += 1024) {
    dia = fma(m.A[i * N + i], m.A[i * N + i], dia);
    rt[i] = noise_root(m.w[i]);
  }
  dia = block_sum<1024>(dia, red);
  // four rows in flight (N is a multiple of 64)
  for (i64 i = threadIdx.x >> 6; i < N; i += 64)
    for (i64 j = threadIdx.x & 63; j < N; j += 64) {
      double v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = m.A[(i + 16 * u) * N + j];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double r = rt[i + 16 * u] * rt[j];
        v[u] = i + 16 * u == j || fabs(v[u]) <= r ? 0.0 : v[u];
        off = fma(v[u], v[u], off);
        large = fabs(v[u]) <= JACOBI_ROW / JACOBI_NOISE * r ? large : 1.0;
      }
    }
  off = block_sum<1024>(off, red);
  large = block_sum<1024>(large, red);
  if (threadIdx.x == 0 && large == 0.0 && off <= JACOBI_TOL * JACOBI_TOL * dia) *m.done = 1;
}

// The rotation of one pair of blocks of round r, accumulated into Q: Jacobi on their
// 64 x 64 submatrix in LDS, 32 disjoint rotations at a time, rows and columns of each
// 2 x 2 block by one thread.  A sweep's first round takes all pairs of the submatrix
// (63 steps), the others only those across the two blocks (32 steps): a sweep then
// takes every pair of the matrix once.  (All pairs in every round: one sweep less of
// 12 at 256 rows, but 441 steps a sweep instead of 255.)  Where the two blocks are the
// whole matrix, up to 30 sweeps at once.  A step is bound by LDS (131 KB of S and W)
// and the chain of the 32 rotations.
constexpr int JB = 32;            // block width
constexpr int JP = 2 * JB;        // order of a pair
constexpr int JPITCH = JP + 1;    // doubles
__global__ __launch_bounds__(1024) void jacobi_pair_kernel(EigArgs a, int r) {
  __shared__ double S[JP * JPITCH], W[JP * JPITCH], cs[JP], red[16];
  __shared__ double w0[JP], rt[JP], part[16][JP];  // weights, their roots
  const EigMode& m = a.m[blockIdx.y];
  const int blocks = m.N / JB;
  if ((int)blockIdx.x >= blocks / 2 || r >= blocks - 1 || *m.done) return;
  const int tid = threadIdx.x;
  int p, q;
  circle_pair(blocks, r, blockIdx.x, p, q);
  const i64 N = m.N;
  for (int e = tid; e < JP * JP; e += 1024) {
    const int i = e / JP, j = e % JP;
    const i64 gi = i < JB ? p * JB + i : q * JB + i - JB, gj = j < JB ? p * JB + j : q * JB + j - JB;
    S[i * JPITCH + j] = m.A[gi * N + gj];
    W[i * JPITCH + j] = i == j ? 1.0 : 0.0;
  }
  double* gw = m.w + (tid < JB ? p * JB + tid : q * JB + tid - JB);  // (tid < JP)
  if (tid < JP) {
    w0[tid] = *gw;
    rt[tid] = noise_root(w0[tid]);
  }
  __syncthreads();
  const int inner = blocks == 2 ? 30 : 1;
  const bool all = r == 0;  // (two blocks have no other round)
  auto pair_of = [&](int rr, int k, int& i, int& j) {
    if (all) {
      circle_pair(JP, rr, k, i, j);
    } else {
      i = k;
      j = JB + ((k + rr) & (JB - 1));
    }
  };
  // the weights after the rotations so far; the steps of one sweep use those before it
  auto weights = [&]() {
    const int j = tid & 63, i = 4 * (tid >> 6);
    double v = 0.0;
#pragma unroll
    for (int e = 0; e < 4; ++e) v = fma(W[(i + e) * JPITCH + j] * W[(i + e) * JPITCH + j], w0[i + e], v);
    part[tid >> 6][j] = v;
    __syncthreads();
    if (tid < JP) {
      v = part[0][j];
#pragma unroll
      for (int e = 1; e < 16; ++e) v += part[e][j];
    }
    return v;  // of the first JP threads
  };
  for (int sweep = 0; sweep < inner; ++sweep) {
    if (sweep > 0) {
      const double wj = weights();
      if (tid < JP) rt[tid] = noise_root(wj);
      __syncthreads();
      double off = 0.0, dia = 0.0, large = 0.0;
      for (int e = tid; e < JP * JP; e += 1024) {
        const double v = S[(e / JP) * JPITCH + e % JP], r = rt[e / JP] * rt[e % JP];
        if (e / JP == e % JP) {
          dia += v * v;
        } else if (!(fabs(v) <= r)) {
          off += v * v;
          large = fabs(v) <= JACOBI_ROW / JACOBI_NOISE * r ? large : 1.0;
        }
      }
      off = block_sum<1024>(off, red);
      dia = block_sum<1024>(dia, red);
      large = block_sum<1024>(large, red);
      if (large == 0.0 && off <= JACOBI_TOL * JACOBI_TOL * dia) break;
    }
    for (int rr = 0; rr < (all ? JP - 1 : JB); ++rr) {
      if (tid < JB) {
        int i, j;
        pair_of(rr, tid, i, j);
        const double apq = S[i * JPITCH + j];
        double c = 1.0, s = 0.0;
        if (!(fabs(apq) <= rt[i] * rt[j])) rotation(S[j * JPITCH + j] - S[i * JPITCH + i], 2.0 * apq, c, s);
        cs[2 * tid] = c;
        cs[2 * tid + 1] = s;
      }
      __syncthreads();
      {
        const int ki = tid >> 5, kj = tid & 31;
        int i0, i1, j0, j1;
        pair_of(rr, ki, i0, i1);
        pair_of(rr, kj, j0, j1);
        const double ci = cs[2 * ki], si = cs[2 * ki + 1], cj = cs[2 * kj], sj = cs[2 * kj + 1];
        const double x00 = S[i0 * JPITCH + j0], x01 = S[i0 * JPITCH + j1], x10 = S[i1 * JPITCH + j0],
                     x11 = S[i1 * JPITCH + j1];
        const double y00 = ci * x00 - si * x10, y01 = ci * x01 - si * x11;
        const double y10 = si * x00 + ci * x10, y11 = si * x01 + ci * x11;
        S[i0 * JPITCH + j0] = cj * y00 - sj * y01;
        S[i0 * JPITCH + j1] = sj * y00 + cj * y01;
        S[i1 * JPITCH + j0] = cj * y10 - sj * y11;
        S[i1 * JPITCH + j1] = sj * y10 + cj * y11;
        // columns j0, j1 of the accumulated rotation: rows ki and ki + 32
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          double* w = W + (ki + 32 * h) * JPITCH;
          const double w0 = w[j0], w1 = w[j1];
          w[j0] = cj * w0 - sj * w1;
          w[j1] = sj * w0 + cj * w1;
        }
      }
      __syncthreads();
    }
  }
  double* out = m.Q + (i64)blockIdx.x * JP * JP;
  for (int e = tid; e < JP * JP; e += 1024) out[e] = W[(e / JP) * JPITCH + e % JP];
  const double wj = weights();
  if (tid < JP) *gw = wj;
}

// A <- J^T A J and V <- V J for the rotations J of round r: workgroup (x, y) owns the
// 64 x 64 tile of A of row pair and column pair (Q_I^T T Q_J), or of 64 rows of V and
// a column pair (T Q_J); tiles are disjoint, so in place.  8 waves, each 16 rows x 32
// columns of the tile, FP64 matrix cores.
__global__ __launch_bounds__(512) void jacobi_update_kernel(EigArgs a, int r) {
  __shared__ double sT[JP * JPITCH], sQ[JP * JPITCH], sP[JP * JPITCH];
  const EigMode& m = a.m[blockIdx.y];
  const int blocks = m.N / JB, pairs = blocks / 2;
  if ((int)blockIdx.x >= 2 * pairs * pairs || r >= blocks - 1 || *m.done) return;
  const bool isV = (int)blockIdx.x >= pairs * pairs;
  const int t = (int)blockIdx.x - (isV ? pairs * pairs : 0), pi = t / pairs, pj = t % pairs;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, q4 = lane >> 4, l16 = lane & 15;
  int rp, rq, cp, cq;
  circle_pair(blocks, r, pi, rp, rq);
  circle_pair(blocks, r, pj, cp, cq);
  if (isV) {  // 64 consecutive rows
    rp = 2 * pi;
    rq = 2 * pi + 1;
  }
  const i64 N = m.N;
  double* M = isV ? m.V : m.A;
  auto grow = [&](int i) { return (i64)(i < JB ? rp * JB + i : rq * JB + i - JB); };
  auto gcol = [&](int j) { return (i64)(j < JB ? cp * JB + j : cq * JB + j - JB); };
  for (int e = tid; e < JP * JP; e += 512) {
    const int i = e / JP, j = e % JP;
    sT[i * JPITCH + j] = M[grow(i) * N + gcol(j)];
    sQ[i * JPITCH + j] = m.Q[(i64)pj * JP * JP + e];
    if (!isV) sP[i * JPITCH + j] = m.Q[(i64)pi * JP * JP + e];
  }
  __syncthreads();
  const int r0 = 16 * (wave >> 1), c0 = 32 * (wave & 1);
  doublex4 acc[2] = {doublex4{0.0, 0.0, 0.0, 0.0}, doublex4{0.0, 0.0, 0.0, 0.0}};
#pragma unroll 4
  for (int kk = 0; kk < JP / 4; ++kk) {
    const double av = sT[(r0 + l16) * JPITCH + 4 * kk + q4];
#pragma unroll
    for (int u = 0; u < 2; ++u)
      acc[u] =
          __builtin_amdgcn_mfma_f64_16x16x4f64(av, sQ[(4 * kk + q4) * JPITCH + c0 + 16 * u + l16], acc[u], 0, 0, 0);
  }
  __syncthreads();
  if (!isV) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) sT[(r0 + 4 * e + q4) * JPITCH + c0 + 16 * u + l16] = acc[u][e];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; ++u) acc[u] = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int kk = 0; kk < JP / 4; ++kk) {
      const double av = sP[(4 * kk + q4) * JPITCH + r0 + l16];  // Q_I^T
#pragma unroll
      for (int u = 0; u < 2; ++u)
        acc[u] =
            __builtin_amdgcn_mfma_f64_16x16x4f64(av, sT[(4 * kk + q4) * JPITCH + c0 + 16 * u + l16], acc[u], 0, 0, 0);
    }
  }
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int e = 0; e < 4; ++e) M[grow(r0 + 4 * e + q4) * N + gcol(c0 + 16 * u + l16)] = acc[u][e];
}

// Workgroup i: if eigenvalue i of the mode is among its top R (descending, ties by
// index), its value and eigenvector, turned so that the first entry of largest
// magnitude is positive.
__global__ __launch_bounds__(256) void eig_select_kernel(EigArgs a) {
  __shared__ int cnt[4];
  __shared__ double bv[4];
  __shared__ int bi[4];
  const EigMode& m = a.m[blockIdx.y];
  const int i = blockIdx.x, n = m.n, tid = threadIdx.x;
  if (i >= n) return;
  const i64 N = m.N;
  const double li = m.A[i * N + i];
  int rk = 0;
  double best = 0.0;  // largest magnitude, its row
  int row = n;
  for (int j = tid; j < n; j += 256) {
    const double lj = m.A[j * N + j];
    rk += (lj > li || (lj == li && j < i)) ? 1 : 0;
    const double v = m.V[j * N + i];
    if (fabs(v) > fabs(best)) {
      best = v;
      row = j;
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    rk += __shfl_xor(rk, off, 64);
    const double ov = __shfl_xor(best, off, 64);
    const int orow = __shfl_xor(row, off, 64);
    if (fabs(ov) > fabs(best) || (fabs(ov) == fabs(best) && orow < row)) {
      best = ov;
      row = orow;
    }
  }
  if ((tid & 63) == 0) {
    cnt[tid >> 6] = rk;
    bv[tid >> 6] = best;
    bi[tid >> 6] = row;
  }
  __syncthreads();
  rk = cnt[0] + cnt[1] + cnt[2] + cnt[3];
  if (rk >= a.R) return;
  best = bv[0];
  row = bi[0];
  for (int w = 1; w < 4; ++w)
    if (fabs(bv[w]) > fabs(best) || (fabs(bv[w]) == fabs(best) && bi[w] < row)) {
      best = bv[w];
      row = bi[w];
    }
  const double sg = best < 0.0 ? -1.0 : 1.0;
  if (tid == 0) m.lam[rk] = li;
  for (int j = tid; j < n; j += 256) m.U[(i64)j * a.R + rk] = sg * m.V[j * N + i];
}

// Nnsvd: for columns j of X_(k) and rank columns r0 .. r0 + 16 of U (n x R):
// z = X_(k)^T u_r; partial[block][r] = (sum of z^2 over z > 0, over z < 0).
constexpr int NN_RC = 16;
__global__ __launch_bounds__(256) void nnsvd_norms_kernel(const float* __restrict__ X, i64 P, i64 I, i64 Q,
                                                          const double* __restrict__ U, int R, int ar,
                                                          double* __restrict__ part) {
  __shared__ double su[256][NN_RC];
  __shared__ double red[2 * NN_RC][4];
  const int tid = threadIdx.x;
  const int r0 = blockIdx.y * NN_RC;
  const i64 J = P * Q;
  const i64 j = (i64)blockIdx.x * 256 + tid;
  const bool live = j < J;
  const i64 p = live ? j / Q : 0, q = live ? j - (j / Q) * Q : 0;
  double z[NN_RC];
#pragma unroll
  for (int u = 0; u < NN_RC; ++u) z[u] = 0.0;
  for (i64 i0 = 0; i0 < I; i0 += 256) {
    for (int e = tid; e < 256 * NN_RC; e += 256) {
      const int ii = e / NN_RC, rr = e % NN_RC;
      su[ii][rr] = (i0 + ii < I && r0 + rr < ar) ? U[(i0 + ii) * R + r0 + rr] : 0.0;
    }
    __syncthreads();
    const i64 iend = std::min<i64>(256, I - i0);
    if (live)
      for (i64 ii = 0; ii < iend; ++ii) {
        const double x = (double)X[(p * I + i0 + ii) * Q + q];
#pragma unroll
        for (int u = 0; u < NN_RC; ++u) z[u] = fma(x, su[ii][u], z[u]);
      }
    __syncthreads();
  }
  // per rank column: sums of positive and negative squares over the block
#pragma unroll
  for (int u = 0; u < NN_RC; ++u) {
    double ps = z[u] > 0.0 ? z[u] * z[u] : 0.0, ns = z[u] < 0.0 ? z[u] * z[u] : 0.0;
    for (int off = 32; off > 0; off >>= 1) {
      ps += __shfl_down(ps, off, 64);
      ns += __shfl_down(ns, off, 64);
    }
    if ((tid & 63) == 0) {
      red[2 * u][tid >> 6] = ps;
      red[2 * u + 1][tid >> 6] = ns;
    }
  }
  __syncthreads();
  if (tid < 2 * NN_RC) {
    const int u = tid >> 1;
    const double s = (red[tid][0] + red[tid][1]) + (red[tid][2] + red[tid][3]);
    if (r0 + u < ar) part[((i64)blockIdx.x * ar + r0 + u) * 2 + (tid & 1)] = s;
  }
}

// One workgroup: the factor (n x R, fp32) of mode k from U (n x R, FP64; columns
// < ar valid), lam, the Nnsvd partials (nblk x ar x 2) and the N(0, 0.01) draws
// rnd (n x (R - ar)) for the columns past ar.
__global__ __launch_bounds__(1024) void svd_init_finish_kernel(const double* __restrict__ U,
                                                               const double* __restrict__ lam, int n, int R, int ar,
                                                               int kind, const double* __restrict__ nn_part, int nblk,
                                                               const float* __restrict__ rnd, float* __restrict__ F) {
  __shared__ double red[16];
  __shared__ double lev_total;
  __shared__ double colv[INIT_RMAX][4];  // Nnsvd: ||u+||^2, ||u-||^2, ||z+||^2, ||z-||^2 per column
  const int tid = threadIdx.x;
  auto block_sum = [&](double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if ((tid & 63) == 0) red[tid >> 6] = v;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < 16; ++w) s += red[w];
    __syncthreads();
    return s;
  };
  if (kind == TENRSO_INIT_LEVERAGE) {
    // l_i = sum_{r < ar} u_ir^2 / ar, normalised by their total when it exceeds
    // f32 epsilon (helpers.rs:329-343)
    double part = 0.0;
    for (int i = tid; i < n; i += 1024) {
      double sc = 0.0;
      for (int r = 0; r < ar; ++r) sc += U[(i64)i * R + r] * U[(i64)i * R + r];
      part += sc / ar;
    }
    const double tot = block_sum(part);
    if (tid == 0) lev_total = tot;
    __syncthreads();
  }
  if (kind == TENRSO_INIT_NNSVD) {
    for (int r = 0; r < ar; ++r) {
      double up = 0.0, un = 0.0;
      for (int i = tid; i < n; i += 1024) {
        const double u = U[(i64)i * R + r];
        if (u > 0.0) up += u * u;
        else un += u * u;
      }
      up = block_sum(up);
      un = block_sum(un);
      double zp = 0.0, zn = 0.0;
      for (int b = tid; b < nblk; b += 1024) {
        zp += nn_part[((i64)b * ar + r) * 2];
        zn += nn_part[((i64)b * ar + r) * 2 + 1];
      }
      zp = block_sum(zp);
      zn = block_sum(zn);
      if (tid == 0) {
        colv[r][0] = up;
        colv[r][1] = un;
        colv[r][2] = zp;
        colv[r][3] = zn;
      }
    }
    __syncthreads();
  }
  for (i64 e = tid; e < (i64)n * R; e += 1024) {
    const int i = (int)(e / R), r = (int)(e - (e / R) * R);
    float out;
    if (r < ar) {
      const double u = U[(i64)i * R + r];
      const double s = sqrt(lam[r] > 0.0 ? lam[r] : 0.0);
      if (kind == TENRSO_INIT_SVD) {
        out = (float)u;
      } else if (kind == TENRSO_INIT_LEVERAGE) {
        double sc = 0.0;
        for (int k = 0; k < ar; ++k) sc += U[(i64)i * R + k] * U[(i64)i * R + k];
        double l = sc / ar;
        if (lev_total > (double)FLT_EPSILON) l /= lev_total;
        out = (float)(u * sqrt(s) * sqrt(l * n));
      } else {
        // ||v+|| = ||z+|| / s (v = z / s); with s == 0 both products are zero
        const double vp = s > 0.0 ? sqrt(colv[r][2]) / s : 0.0, vn = s > 0.0 ? sqrt(colv[r][3]) / s : 0.0;
        const double pp = sqrt(colv[r][0]) * vp, np = sqrt(colv[r][1]) * vn;
        if (pp >= np) out = (float)((u > 0.0 ? u : 0.0) * sqrt(s * pp));
        else out = (float)((u > 0.0 ? 0.0 : -u) * sqrt(s * np));
      }
    } else {
      const float d = rnd[(i64)i * (R - ar) + (r - ar)];
      if (kind == TENRSO_INIT_SVD) {
        out = d;
      } else if (kind == TENRSO_INIT_NNSVD) {
        out = fabsf(d);
      } else {
        double sc = 0.0;
        for (int k = 0; k < ar; ++k) sc += U[(i64)i * R + k] * U[(i64)i * R + k];
        double l = ar > 0 ? sc / ar : 0.0;
        if (lev_total > (double)FLT_EPSILON) l /= lev_total;
        out = (float)(d * l);
      }
    }
    F[e] = out;
  }
}

}  // namespace

int cp_init_svd(tenrso_ctx* ctx, const float* X, int nd, const i64* shape, i64 R, int kind, uint64_t seed,
                float* const* F) {
  if (kind != TENRSO_INIT_SVD && kind != TENRSO_INIT_NNSVD && kind != TENRSO_INIT_LEVERAGE) {
    set_error("unknown initialisation kind %d", kind);
    return TENRSO_ERR_INVALID_ARGUMENT;
  }
  if (nd < 1 || nd > MAXD) {
    set_error("tensors with %d modes are not supported", nd);
    return TENRSO_ERR_UNSUPPORTED;
  }
  if (R <= 0 || R > INIT_RMAX) {
    set_error("rank %lld outside the on-device SVD initialisation bound 1..%d", (long long)R, INIT_RMAX);
    return TENRSO_ERR_UNSUPPORTED;
  }
  for (int k = 0; k < nd; ++k) {
    if (shape[k] > EIG_NMAX) {
      set_error("mode %d of size %lld exceeds the on-device SVD initialisation bound %d", k, (long long)shape[k],
                EIG_NMAX);
      return TENRSO_ERR_UNSUPPORTED;
    }
    if (shape[k] <= 0) {
      set_error("mode %d is empty", k);
      return TENRSO_ERR_DEVICE;
    }
  }
  // what depends on a mode: J columns of its unfolding, the splits of its Gram
  // (about 1024 workgroups, at most 64 MiB of partials), the layout of its buffers
  struct Mode {
    i64 P, I, Q, J, nt, splits, nn_blk, oA, oQ, oW, oU, oNN, oR;
    int ar;
  } md[MAXD];
  i64 totA = 0, totQ = 0, totN = 0, totU = 0, totNN = 0, totR = 0, part = 0;
  EigArgs ea{};
  ea.R = (int)R;
  for (int k = 0; k < nd; ++k) {
    Mode& m = md[k];
    m.P = m.Q = 1;
    for (int j = 0; j < k; ++j) m.P *= shape[j];
    for (int j = k + 1; j < nd; ++j) m.Q *= shape[j];
    m.I = shape[k];
    m.J = m.P * m.Q;
    m.ar = (int)std::min<i64>(R, std::min<i64>(m.I, m.J));
    m.nt = (m.I + GT - 1) / GT;
    const i64 ntp = m.nt * (m.nt + 1) / 2;
    m.splits = std::max<i64>(1, std::min<i64>((1024 + ntp - 1) / ntp, (m.J + 4 * GK - 1) / (4 * GK)));
    m.splits = std::max<i64>(1, std::min<i64>(m.splits, (64ll << 20) / (m.I * m.I * 8)));
    part = std::max(part, m.splits * m.I * m.I);
    const i64 N = (m.I + JP - 1) / JP * JP;
    ea.m[k].n = (int)m.I;
    ea.m[k].N = (int)N;
    m.oA = totA;
    totA += N * N;
    m.oQ = totQ;
    totQ += N / JP * JP * JP;
    m.oW = totN;
    totN += N;
    m.oU = totU;
    totU += m.I * R + R;
    m.nn_blk = (m.J + 255) / 256;
    m.oNN = totNN;
    totNN += kind == TENRSO_INIT_NNSVD ? m.nn_blk * m.ar * 2 : 0;
    m.oR = totR;
    totR += m.I * (R - m.ar);
  }
  void *pA, *pV, *pPart, *pW;
  TENRSO_TRY(ctx_buffer(ctx, SLOT_EIG_A, (size_t)(totA + totQ) * 8, &pA));
  TENRSO_TRY(ctx_buffer(ctx, SLOT_EIG_V, (size_t)(totA + totN) * 8 + MAXD * sizeof(int), &pV));
  TENRSO_TRY(ctx_buffer(ctx, SLOT_EIG_PART, (size_t)part * 8, &pPart));
  TENRSO_TRY(ctx_buffer(ctx, SLOT_EIG_W, (size_t)(totU + totNN) * 8 + (size_t)totR * 4 + 16, &pW));
  float* rnd = (float*)((double*)pW + totU + totNN);
  int maxN = 0;
  for (int k = 0; k < nd; ++k) {
    const Mode& m = md[k];
    EigMode& e = ea.m[k];
    e.A = (double*)pA + m.oA;
    e.Q = (double*)pA + totA + m.oQ;
    e.V = (double*)pV + m.oA;
    e.w = (double*)pV + totA + m.oW;
    e.done = (int*)((double*)pV + totA + totN) + k;
    e.U = (double*)pW + m.oU;
    e.lam = e.U + m.I * R;
    maxN = std::max(maxN, e.N);
    hipLaunchKernelGGL(unfold_gram_partial_kernel, dim3((unsigned)(m.nt * (m.nt + 1) / 2), (unsigned)m.splits),
                       dim3(256), 0, ctx->stream, X, m.P, m.I, m.Q, (int)m.nt, (int)m.splits, (double*)pPart);
    TENRSO_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(unfold_gram_reduce_kernel, dim3((unsigned)((i64)e.N * e.N / 256)), dim3(256), 0, ctx->stream,
                       (const double*)pPart, (int)m.splits, e);
    TENRSO_HIP_TRY(hipGetLastError());
  }
  // A mode that has converged skips what is queued, 2-3 us a launch.  The host looks
  // after JACOBI_FIRST sweeps and then after each (about 20 us); where the call is being
  // captured it cannot, and all sweeps are queued.  Two blocks are solved in one sweep.
  const int pairs = maxN / JP, rounds = maxN / JB - 1;
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  TENRSO_HIP_TRY(hipStreamIsCapturing(ctx->stream, &capture));
  const bool look = capture == hipStreamCaptureStatusNone;
  for (int sweep = 0; sweep <= JACOBI_SWEEPS; ++sweep) {
    hipLaunchKernelGGL(jacobi_check_kernel, dim3((unsigned)nd), dim3(1024), 0, ctx->stream, ea);
    TENRSO_HIP_TRY(hipGetLastError());
    if (look && sweep >= (rounds == 1 ? 1 : JACOBI_FIRST)) {
      int done[MAXD];
      TENRSO_HIP_TRY(hipMemcpyAsync(done, ea.m[0].done, nd * sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
      TENRSO_HIP_TRY(hipStreamSynchronize(ctx->stream));
      if (std::all_of(done, done + nd, [](int d) { return d != 0; })) break;
    }
    if (sweep == JACOBI_SWEEPS) break;
    for (int r = 0; r < rounds; ++r) {
      hipLaunchKernelGGL(jacobi_pair_kernel, dim3((unsigned)pairs, (unsigned)nd), dim3(1024), 0, ctx->stream, ea, r);
      hipLaunchKernelGGL(jacobi_update_kernel, dim3((unsigned)(2 * pairs * pairs), (unsigned)nd), dim3(512), 0,
                         ctx->stream, ea, r);
    }
    TENRSO_HIP_TRY(hipGetLastError());
  }
  hipLaunchKernelGGL(eig_select_kernel, dim3((unsigned)maxN, (unsigned)nd), dim3(256), 0, ctx->stream, ea);
  TENRSO_HIP_TRY(hipGetLastError());
  std::mt19937_64 rng(seed);
  std::normal_distribution<double> noise(0.0, 0.01);  // helpers.rs: Normal::new(0.0, 0.01)
  for (int k = 0; k < nd; ++k) {
    const Mode& m = md[k];
    const EigMode& e = ea.m[k];
    double* nn = (double*)pW + totU + m.oNN;
    float* draws = rnd + m.oR;
    if (kind == TENRSO_INIT_NNSVD && m.ar > 0) {
      hipLaunchKernelGGL(nnsvd_norms_kernel, dim3((unsigned)m.nn_blk, (unsigned)((m.ar + NN_RC - 1) / NN_RC)), dim3(256),
                         0, ctx->stream, X, m.P, m.I, m.Q, (const double*)e.U, (int)R, m.ar, nn);
      TENRSO_HIP_TRY(hipGetLastError());
    }
    if (m.ar < R) {
      std::vector<float> h((size_t)m.I * (R - m.ar));
      for (auto& v : h) v = (float)noise(rng);
      TENRSO_HIP_TRY(hipMemcpyAsync(draws, h.data(), h.size() * 4, hipMemcpyHostToDevice, ctx->stream));
      TENRSO_HIP_TRY(hipStreamSynchronize(ctx->stream));  // h leaves scope
    }
    hipLaunchKernelGGL(svd_init_finish_kernel, dim3(1), dim3(1024), 0, ctx->stream, (const double*)e.U,
                       (const double*)e.lam, (int)m.I, (int)R, m.ar, kind, (const double*)nn, (int)m.nn_blk,
                       (const float*)draws, F[k]);
    TENRSO_HIP_TRY(hipGetLastError());
  }
  return TENRSO_OK;
}

}  // namespace tenrso
