// als_job_wide.hpp -- the ALS job of ranks JOB_NE + 1 .. WIDE_NE: the steps of
// als_job.hpp (the fit, Gamma_n plus regularisation, its inverse with the ridge
// retry of cp/helpers.rs:477-490) as one workgroup of 512 threads, on its own or as
// workgroup 0 of an MTTKRP launch.
//
// The 128 x 128 symmetric matrix (the identity outside R x R) is held as its upper
// triangle of 16 x 16 tiles in the accumulators of v_mfma_f64_16x16x4f64: a wave
// owns the strip of rows 16 st .. + 15 and its tiles u = 0 .. 7 - st of columns
// 16 (st + u) ..; lane l, element e of a tile holds
//   A[16 st + 4 e + l/16][16 (st + u) + l%16].
// Waves w and w + 4, which share a SIMD, own strips w and 7 - w: nine tiles a SIMD.
#pragma once
#include "als_job.hpp"
#include "cp_linalg.hpp"

namespace tenrso {

constexpr int WIDE_THREADS = 512;
// LDS (doubles): [2][4][128] pivot rows, [2][16] pivot-block inverses, 2 x 8 wave
// sums, one flag, and a place per lane for stores that a lane does not make
constexpr int WIDE_ROW = 0, WIDE_PINV = 2 * 4 * WIDE_NE, WIDE_RED = WIDE_PINV + 2 * 16, WIDE_FLAG = WIDE_RED + 16,
              WIDE_NONE = WIDE_FLAG + 2;
constexpr int WIDE_LDS_BYTES = (WIDE_NONE + 64) * 8;

__device__ __forceinline__ double wide_block_sum(double v, double* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int w = 0; w < WIDE_THREADS / 64; ++w) s += red[w];
  return s;
}

// Inverse of the 4 x 4 pivot block at lds[pb] (rows of stride WIDE_NE) by one wave,
// into lds[pi], the block itself replaced by the identity.  Every lane sweeps the
// symmetric block's upper triangle, one scalar pivot after another (the sweep of
// pivot p: a_ij -= a_ip a_pj / a_pp, a_ip /= a_pp, a_pp = -1 / a_pp, which ends with
// minus the inverse).  A pivot that is not positive and finite sets the flag.  Cofactors
// over the determinant were shorter by 0.1 us a step, but their error grows with the
// cube of the block's condition, not with the condition itself: factors with four
// collinear columns (condition 1e7) came out with an inverse off by 1e-3 instead of
// 1e-9, and at 1e9 the determinant's sign was noise.
__device__ __forceinline__ void wide_invert_pivot(double* lds, int pb, int pi) {
  const int lane = threadIdx.x & 63, lr = (lane >> 2) & 3, lc = lane & 3;
  const double* Pb = lds + pb;
  double p[4][4];  // upper triangle
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int k = i; k < 4; ++k) p[i][k] = Pb[i * WIDE_NE + k];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  const int none = WIDE_NONE + lane;
  lds[lane < 16 ? pb + lr * WIDE_NE + lc : none] = lr == lc ? 1.0 : 0.0;
  bool good = true;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    good = good & (p[k][k] > 0.0) & (p[k][k] <= DBL_MAX);
    const double d = job_recip(p[k][k]);
    double b[4], t[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      b[i] = i < k ? p[i][k] : p[k][i];
      t[i] = b[i] * d;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int m = i; m < 4; ++m)
        if (i != k && m != k) p[i][m] = fma(-t[i], b[m], p[i][m]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i < k) p[i][k] = t[i];
      if (i > k) p[k][i] = t[i];
    }
    p[k][k] = -d;
  }
  // lane (r, c) stores entry (r, c)
  double v = p[0][0];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int k = i; k < 4; ++k) v = (lr == i && lc == k) || (lr == k && lc == i) ? p[i][k] : v;
  lds[lane < 16 ? pi + lr * 4 + lc : none] = -v;
  lds[((lane < 16) & !good) ? WIDE_FLAG : none] = 1.0;
}

// Block Gauss-Jordan inverse on the FP64 matrix cores: the elimination of
// job_block_gj (als_job.hpp has the formulas) on the upper triangle, R/4 steps of
// one barrier each.  Step s eliminates rows and columns J = {4s .. 4s+3} of strip
// s/4.  The rows J of the next step are published whole, with the identity in the
// pivot columns (their part of W is P^-1): the pivot's wave holds them from its
// diagonal tile on; the columns before it lie transposed in the tiles of the strips
// above, whose rows are all eliminated, so there A[J][c] = -A[c][J].  What a step
// replaces (rows and columns J) is zeroed by the wave that publishes it.  The
// pivot's wave updates its diagonal tile first and inverts the next pivot block
// beside its other MFMAs (s_setprio: ahead of the other wave of its SIMD).  False
// if a pivot block is not positive definite.
// Bound: nine tiles a SIMD and step (64 + 16 cycles each: 720 cycles), 11 us over
// the 32 steps of rank 128 at 2.1 GHz, and the chain of a step (barrier, LDS, W,
// the diagonal tile, publishing and inverting the pivot): 0.87 us a step.  The job
// alone takes 37 us at rank 128 and 24 us at rank 66; one FMA pass a step over the
// full matrix in 1024 threads' registers took 101 us at rank 128.
template <int ST>
__device__ __forceinline__ bool wide_block_gj(doublex4 (&acc)[8 - ST], int R, double* lds) {
  constexpr int NE = WIDE_NE, NU = 8 - ST;
  double* rowb = lds + WIDE_ROW;
  const double* pinv = lds + WIDE_PINV;
  const int lane = threadIdx.x & 63, q = lane >> 4, j = lane & 15;
  const int steps = (R + 3) / 4;
  auto zero_cols = [](doublex4& t, bool z) {
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] = z ? 0.0 : t[e];
  };
  if (threadIdx.x == 0) lds[WIDE_FLAG] = 0.0;
  __syncthreads();
  if constexpr (ST == 0) {
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      rowb[q * NE + 16 * u + j] = acc[u][0];
      acc[u][0] = 0.0;
    }
    zero_cols(acc[0], j < 4);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    wide_invert_pivot(lds, WIDE_ROW, WIDE_PINV);
  }
  for (int ps = 0; 4 * ps < steps; ++ps) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int s = 4 * ps + e, s1 = s + 1;
      if (s >= steps) break;
      const int e1 = (e + 1) & 3, ps1 = e == 3 ? ps + 1 : ps;
      const double* Rw = rowb + (e & 1) * 4 * NE;
      double* Rn = rowb + (e1 & 1) * 4 * NE;
      __syncthreads();
      const double pa = pinv[(e & 1) * 16 + (lane & 3) * 4 + q];  // P^-1[l & 3][l >> 4]
      const double rown = Rw[q * NE + 16 * ST + j];
      double rb[NU];
#pragma unroll
      for (int u = 0; u < NU; ++u) rb[u] = Rw[q * NE + 16 * (ST + u) + j];
      // -A[16 ST + j][J_q]; +I on the pivot rows
      double aop = 16 * ST + j < 4 * s ? rown : -rown;
      aop = ((ST == ps) & ((j >> 2) == e)) ? ((j & 3) == q ? 1.0 : 0.0) : aop;
      const bool col1 = (j >> 2) == e1;  // a pivot column of the next step's tile
      auto tile = [&](int u) {
        const double wv = __builtin_amdgcn_mfma_f64_4x4x4f64(pa, rb[u], 0.0, 0, 0, 0);
        acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(aop, wv, acc[u], 0, 0, 0);
      };
      const bool next = ps1 == ST && s1 < steps;
      if (next) __builtin_amdgcn_s_setprio(3);
      tile(0);
      if (next) {
        Rn[q * NE + 16 * ST + j] = acc[0][e1];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        wide_invert_pivot(lds, WIDE_ROW + (e1 & 1) * 4 * NE + 4 * s1, WIDE_PINV + (e1 & 1) * 16);
      }
#pragma unroll
      for (int u = 1; u < NU; ++u) tile(u);
      if (next) {
#pragma unroll
        for (int u = 1; u < NU; ++u) Rn[q * NE + 16 * (ST + u) + j] = acc[u][e1];
#pragma unroll
        for (int u = 0; u < NU; ++u) acc[u][e1] = 0.0;
        zero_cols(acc[0], col1);
        __builtin_amdgcn_s_setprio(0);
      }
      if (ps1 > ST && s1 < steps) {
        // Left to itself the compiler turns the choice of tile below into one indexed
        // register read (s_set_gpr_idx_on, v_mov_b32 from the first tile's registers),
        // and the wait that a read of an FP64 MFMA's result needs is then counted from
        // the first tile's MFMA, not from the last one's: a last tile read that way
        // came out stale.  Tied to the accumulators, the wait stands here for all of
        // them, and the reads name their registers, as those of the pivot's wave above
        // do anyway.
#pragma unroll
        for (int u = 1; u < NU; ++u) asm volatile("" : "+v"(acc[u]));
        asm volatile("s_nop 15\n\ts_nop 15" : "+v"(acc[NU - 1]));
        const int pub = WIDE_ROW + (e1 & 1) * 4 * NE + (j & 3) * NE + 16 * ST + q;
#pragma unroll
        for (int u = 1; u < NU; ++u) {
          if (ST + u == ps1) {
#pragma unroll
            for (int e2 = 0; e2 < 4; ++e2) lds[col1 ? pub + 4 * e2 : WIDE_NONE + lane] = -acc[u][e2];
            zero_cols(acc[u], col1);
          }
        }
      }
    }
  }
  __syncthreads();
  const bool ok = lds[WIDE_FLAG] == 0.0;
  __syncthreads();  // every thread has read the flag before a retry resets it
  return ok;
}

// The job of the wave that owns strip ST.
template <int ST>
__device__ __forceinline__ void als_job_wide_strip(const AlsJob& a, double* lds) {
  constexpr int st = ST, NU = 8 - ST;
  const int R = a.R;
  const int q = (threadIdx.x & 63) >> 4, j = threadIdx.x & 15;
  const int row0 = 16 * st + q;  // element e of a tile is row row0 + 4 e, tile u column 16 (st + u) + j
  double ipv = 0.0;
  if (a.do_fit)
    for (int b = threadIdx.x; b < a.nblk; b += WIDE_THREADS) ipv += a.ip_part[b];
  // gam = hadamard of the Grams k != skip; entries outside R x R are 0
  doublex4 gam[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) gam[u] = doublex4{1.0, 1.0, 1.0, 1.0};
  double rec = 0.0;
  // the last pass (with the fit only): ||Xhat||^2 = sum_{r,s} prod_k G_k[r,s], that is
  // gam times the Gram of mode skip; tiles off the diagonal count twice
  const int last = a.do_fit ? a.nd : a.nd - 1;
#pragma unroll 1
  for (int k = 0; k <= last; ++k) {
    const bool fit = k == a.nd;
    if (k == a.skip) continue;
    const double* Gk = a.G + (i64)(fit ? (a.skip < 0 ? 0 : a.skip) : k) * R * R;
    const bool ones = fit && a.skip < 0;  // gam has every mode
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int col = 16 * (st + u) + j;
      doublex4 g;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = row0 + 4 * e;
        g[e] = (i < R && col < R) ? Gk[i * R + col] : 0.0;
        if (ones) g[e] = (i < R && col < R) ? 1.0 : 0.0;
      }
      if (fit) {
        const double t = (gam[u][0] * g[0] + gam[u][1] * g[1]) + (gam[u][2] * g[2] + gam[u][3] * g[3]);
        rec += u == 0 ? t : 2.0 * t;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) gam[u][e] *= g[e];
      }
    }
  }
  if (a.do_fit) {
    const double recon = wide_block_sum(rec, lds + WIDE_RED);
    const double ip = wide_block_sum(ipv, lds + WIDE_RED + 8);
    if (threadIdx.x == 0) {
      double blk[JOB_SC_STAMP];
#pragma unroll
      for (int i = 0; i < JOB_SC_STAMP; ++i) blk[i] = a.scal[i];
      const double nx = blk[JOB_SC_NORM_X];
      const double err_sq = nx + recon - 2.0 * ip;
      const double err = sqrt(err_sq > 0.0 ? err_sq : 0.0);
      double fit = 1.0 - err / sqrt(nx);
      fit = fit < 0.0 ? 0.0 : (fit > 1.0 ? 1.0 : fit);
      blk[JOB_SC_FIT] = fit;
      blk[JOB_SC_IP] = ip;
      blk[JOB_SC_RECON] = recon;
      a.scal[JOB_SC_FIT] = fit;
      a.scal[JOB_SC_IP] = ip;
      a.scal[JOB_SC_RECON] = recon;
      if (a.host) {
#pragma unroll
        for (int i = 0; i < JOB_SC_STAMP; ++i) a.host[i] = blk[i];
        __threadfence_system();
        a.host[JOB_SC_STAMP] = a.stamp;
      }
    }
  }
  if (a.gate) {
    __syncthreads();  // every thread has its Grams
    if (threadIdx.x == 0) __hip_atomic_store(a.gate, a.gate_stamp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (a.skip < 0) return;
  // Gamma waits in Winv for the ridge retry (each thread rereads its own entries)
  double* wp = a.Winv + row0 * WIDE_NE + 16 * st + j;
#pragma unroll
  for (int u = 0; u < NU; ++u) {
#pragma unroll
    for (int e = 0; e < 4; ++e) wp[4 * e * WIDE_NE + 16 * u] = gam[u][e];
  }
  bool ok = false;
  int path = 0;
  for (;;) {
    const double ridge = path ? (double)FLT_EPSILON * (double)(10 * R) : 0.0;
    const bool band = ridge > 0.0 || a.tik_order > 0 || a.l2 > 0.0;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int col = 16 * (st + u) + j;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = row0 + 4 * e;
        if (!(i < R && col < R)) gam[u][e] = i == col ? 1.0 : 0.0;
        else if (band) gam[u][e] += job_reg(a, i, col, ridge);
      }
    }
    ok = wide_block_gj<ST>(gam, R, lds);
    if (ok || path) break;
    path = 1;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
#pragma unroll
      for (int e = 0; e < 4; ++e) gam[u][e] = wp[4 * e * WIDE_NE + 16 * u];
    }
  }
  if (!ok) path = 2;
  // both triangles
  double* wt = a.Winv + (16 * st + j) * WIDE_NE + row0;
#pragma unroll
  for (int u = 0; u < NU; ++u) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const double v = ok ? gam[u][e] : 0.0;
      wp[4 * e * WIDE_NE + 16 * u] = v;
      if (u > 0) wt[16 * u * WIDE_NE + 4 * e] = v;
    }
  }
  if (threadIdx.x == 0 && a.scal) {
    const double prev = a.scal[a.status_slot];
    a.scal[a.status_slot] = a.status_reset ? (double)path : fmax(prev, (double)path);
  }
}

// The whole job; `lds` must hold WIDE_LDS_BYTES (16-byte aligned).  All 512 threads
// of the workgroup must call it.  Every strip has code of its own (its tiles are
// register indices), with the same barriers.
__device__ __forceinline__ void als_job_wide_run(const AlsJob& a, double* lds) {
  switch (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) {
    case 0: als_job_wide_strip<0>(a, lds); break;
    case 1: als_job_wide_strip<1>(a, lds); break;
    case 2: als_job_wide_strip<2>(a, lds); break;
    case 3: als_job_wide_strip<3>(a, lds); break;
    case 4: als_job_wide_strip<7>(a, lds); break;
    case 5: als_job_wide_strip<6>(a, lds); break;
    case 6: als_job_wide_strip<5>(a, lds); break;
    default: als_job_wide_strip<4>(a, lds); break;
  }
}

}  // namespace tenrso
