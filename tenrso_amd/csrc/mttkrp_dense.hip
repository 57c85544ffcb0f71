// mttkrp_dense.hip -- dense mode-n MTTKRP for gfx950 (MI355X).
//
// Contract of tenrso_kernels::mttkrp (tenrso-kernels/src/mttkrp.rs:74-146):
//   V[i, r] = sum_j X_(n)[i, j] * KR[j, r]
// where X_(n) is the forward-order unfolding (mttkrp.rs:149-177) and KR the
// forward-order Khatri-Rao product of the other factors (mttkrp.rs:182-240).
//
// Design (no unfolding copy, no materialised KR):
//   * X is viewed in place as [P, I, Q] (P = prod of modes before n, Q = after).
//     The contraction index j = (p, q) runs over the other modes in forward order,
//     so j = p*Q + q and X[p, i, q] sits at (p*I + i)*Q + q.
//   * j = (slow, k): k runs over the fastest other mode, slow over the rest, and
//     KR[j, r] = PRE[slow, r] * FAST[k, r], where FAST is the factor of the
//     fastest other mode and PRE the forward KR of the remaining other modes (a
//     factor itself for 3-way tensors).  A workgroup stages a window of FAST,
//     transposed to [r][k], in LDS once, contracts
//     T[i, r] = sum_k X[.., i, .., k] FAST[k, r] per slow index and adds
//     PRE[slow, r] T[i, r] into its accumulator.  No Khatri-Rao row is ever
//     written to memory.
//   * Rows i are the MFMA M dimension, rank columns r the N dimension, j the K
//     dimension, in v_mfma_f32_16x16x32_bf16: an fp32 tensor as exact triples of
//     bf16 (mttkrp_x3_kernel.hpp), a bf16 tensor as it is (here).  For q-contiguous X
//     (mode < N-1, "case A") each lane loads 8 consecutive j straight from HBM; for
//     the last mode (Q == 1, "case B") lanes run along i, which is contiguous, and
//     each lane loads its 8 j of two rows (bf16: four).
//   * Workgroups split j; each writes an [I_tile x R] fp32 partial, summed in a
//     fixed order (FP64) by reduce_partials or by the ALS solve kernel.  No float
//     atomics: results are run-to-run deterministic.
#include <algorithm>

#include "mttkrp_tile.hpp"
#include "mttkrp_x3.hpp"

namespace tenrso {

// ---------------------------------------------------------------------------
// BF16 MFMA kernel (v_mfma_f32_16x16x32_bf16).  The work split and the T-then-PRE
// contraction of the fp32 kernel (mttkrp_x3_kernel.hpp), FP32 accumulation.  X
// enters as it is.
//   XL 0, 1, 4 (16-byte aligned rows; case A): whole windows, masked windows, a
// zero-padded copy.  One 16-byte load of 8 consecutive j per lane, row and k-step; the
// FAST window enters as a bf16 hi + lo pair (two MFMAs per step).
//   XL 3 (any size and alignment; both cases) and case B (the last mode; XL 0 for I a
// multiple of 4 and an 8-byte aligned X): the FAST window as the exact triple of each
// fp32 value, so the products are those of fp32 arithmetic, as they are in the
// one-thread-an-output kernel that served such calls (2000 us at 19x69x32x75 rank 21;
// 70 us here).  Vectors are loaded unaligned, elements past the window's end (the next
// row's) are masked, except where the load would pass the end of X.  As in the fp32
// kernel a tile that is not finite, or whose values are too small for their low parts,
// is formed again with the fp32 instruction.
//   Case B: 64 rows a workgroup, lanes along i; each lane loads four rows (8 bytes) of
// its 8 j, a full 128-byte line per j and 16 lanes, and byte permutes turn the 8 x 4
// block into four A operands.  (A copy of X with the last mode in front took 43 us of
// the 64 of a 512x512x128 rank 64 last mode; this form takes 20.)
// ---------------------------------------------------------------------------
template <int NT, int WAVES, int KS, int KWMAX, bool CASE_B, bool WV, int XL>
__global__ __launch_bounds__(WAVES * 64) void mttkrp_bf16_mfma(const uint16_t* __restrict__ X, KernArgs a,
                                                               float* __restrict__ partial, AlsJob job, int has_job) {
  constexpr int MT = CASE_B ? 4 : 2, NBUF = CASE_B ? 3 : 4;
  constexpr bool EXACT = CASE_B || XL == 3;  // FAST as triples
  constexpr int KB = 32 * KS, PITCH = KWMAX + 8, RT = 16 * NT, NTH = WAVES * 64, ROWS = 16 * MT;
  constexpr int LDS_WIN = (EXACT ? 3 : 2) * RT * PITCH * 2, LDS_RED = MT * NT * WAVES * 64 * 16;
  constexpr int LDS_B = LDS_WIN > LDS_RED ? LDS_WIN : LDS_RED;
  constexpr int LDS_BYTES = CASE_B || LDS_B > JOB_LDS_BYTES ? LDS_B : JOB_LDS_BYTES;
  static_assert(!CASE_B || KS == 1, "case B takes blocks of 32");
  __shared__ __attribute__((aligned(16))) float smem[LDS_BYTES / 4];
  __shared__ float wmin[WAVES];  // smallest magnitude of the window values that each wave stages
  __shared__ int redo;           // a wave asks for the fp32 form
  if constexpr (!CASE_B) {  // the BF16 ALS contracts its last mode in fp32
    static_assert(NTH % JOB_THREADS == 0, "the ALS job runs on the first 256 threads");
    if (has_job && blockIdx.x == 0) {
      // the job's workgroup: waves past the job's four end at once (a barrier
      // no longer waits for an ended wave); with one such workgroup per CU the
      // job has its CU to itself
      if (threadIdx.x < JOB_THREADS) als_job_run(job, reinterpret_cast<double*>(smem));
      return;
    }
    if (has_job && job.gate) {
      // start gate: wait (a bounded number of polls) until the job has its Grams
      if (threadIdx.x == 0) {
        for (int it = 0; it < JOB_GATE_POLLS; ++it) {
          if (__hip_atomic_load(job.gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == job.gate_stamp) break;
          __builtin_amdgcn_s_sleep(8);
        }
      }
      __syncthreads();
    }
  }
  const int tile = a.tile0 + (int)blockIdx.x - (!CASE_B && has_job ? 1 : 0);
  const int xt = tile % a.rtiles;
  uint16_t* sHi = reinterpret_cast<uint16_t*>(smem);
  uint16_t* sLo = sHi + RT * PITCH;
  uint16_t* sLo2 = sLo + RT * PITCH;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: scalar schedule and addresses
  const int g = lane >> 4, c = lane & 15;
  const int split = tile / a.rtiles;
  const int w = split % a.nwin;
  const int ss = split / a.nwin;
  // balanced split of the slow range: the first slow_rem splits take one more
  const i64 s_lo = uniform_i64((i64)ss * a.slow_q + (ss < a.slow_rem ? ss : a.slow_rem));
  const i64 s_hi = s_lo + a.slow_q + (ss < a.slow_rem ? 1 : 0);
  // rows of this window that exist
  const int kv = XL == 0 ? a.kw : (int)min((i64)a.kw, a.fast_size - (i64)w * a.kw);
  const int nkb = XL == 0 ? a.kw / KB : (kv + KB - 1) / KB;
  // the workgroup's blocks (slow index, then block within it) in WAVES contiguous,
  // balanced ranges: with 9 slow indices of 4 blocks, 9 blocks per wave rather
  // than 12 for one wave and 8 for the others
  const i64 nblk_wg = (s_hi - s_lo) * nkb;
  const i64 wb0 = uniform_i64(wave * nblk_wg / WAVES), wb1 = (wave + 1) * nblk_wg / WAVES;
  const int T = __builtin_amdgcn_readfirstlane((int)(wb1 - wb0));  // blocks of this wave
  const i64 wq = whole_slow(wb0, nkb);
  const int wr = (int)(wb0 - wq * nkb);  // its first: block wr of slow index s_lo + wq
  const i64 row_base = (i64)xt * ROWS;
  if (tid == 0) redo = 0;

  FastWindow<RT, NTH, KWMAX> fw;  // window loads before the X blocks
  stage_window_load<WV>(fw, a, w, kv);

  floatx4 acc[MT][NT], Tacc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      acc[mt][nt] = floatx4{0.f, 0.f, 0.f, 0.f};
      Tacc[mt][nt] = floatx4{0.f, 0.f, 0.f, 0.f};
    }

  // case A: x[mt][ks], 8 j of a row; case B: the 8 j, four rows each
  struct Buf {
    uint32x4 x[CASE_B ? 4 : MT][KS];
    float pre[NT];
    int kb;
    uint32_t okm;  // XL 1: bit ks set where the vector of k-step ks lies below kv
  };

  // per-lane element offsets, fixed for the whole loop; the per-block part of
  // every address is wave-uniform
  // Case A, XL 3: eights of a block that are read.  In a window of one block those past
  // its end are not: their lanes load what the last ones do.
  const int eights = XL == 3 && nkb == 1 ? (kv + 7) / 8 : KB / 8, gl = min(g, eights - 1);
  i64 loff[MT];
  int shift = 0;  // case B: bits by which the lane's rows lie above the loaded four
  if constexpr (!CASE_B) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const i64 rr = row_base + 16 * mt + c;
      loff[mt] = (rr < a.I ? rr : a.I - 1) * a.Q + 8 * gl;
    }
  } else {
    const i64 rr = row_base + MT * c, top = a.I > MT ? a.I - MT : 0;
    loff[0] = (i64)(8 * g) * a.I + (rr < top ? rr : top);
    if (XL != 0 && rr > top && rr < a.I) shift = 16 * (int)(rr - top);
  }
  // XL 3: a block starting past `lim` would read past the end of X
  i64 lim = 0;
  if constexpr (XL == 3) {
    const i64 last = (row_base + ROWS < a.I ? row_base + ROWS : a.I) - 1;
    lim = uniform_i64(CASE_B ? a.total - (i64)(KB - 1) * a.I - (a.I > MT ? a.I : MT)
                             : a.total - last * a.Q - 8 * eights);
  }
  // PRE column of each lane: columns past rcount read column r0 (those
  // accumulator columns are never stored)
  const bool has_pre = a.pre != nullptr;
  const float* pre_base = has_pre ? a.pre : kPreOnes;
  const i64 pre_stride = has_pre ? a.R : 0;
  int poff[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) poff[nt] = (has_pre ? a.r0 : 0) + (16 * nt + c < a.rcount ? 16 * nt + c : 0);

  BlockCursor<KB, CASE_B> cur(a, s_lo + wq, w, nkb, wr);

  auto load = [&](int t, Buf& b) {
    b.kb = cur.kb;
    // (whole windows: PRE is loaded again only where the slow index changes; at rank 64
    // four loads a block beside X's four cost a BF16 ALS of 256^3 1 to 2 %)
    const float* prow = pre_base + opaque_uniform<CASE_B || XL != 0>(cur.slow * pre_stride);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) b.pre[nt] = prow[poff[nt]];
    const bool live = t < T;  // past the end: one cache line at X (see the fp32 kernel)
    const i64 off = opaque_uniform(live ? cur.offset(a) : 0);
    const uint16_t* ubase = X + off;
    bool inside = true;  // uniform
    if constexpr (XL == 3) inside = live ? off <= lim : a.total >= 8;
    // XL 1: vectors at k >= kv (a multiple of 8) are loaded from X instead and zeroed
    b.okm = 0xffu;
    if constexpr (XL == 1) {
      b.okm = 0;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) b.okm |= (live && b.kb * KB + 32 * ks + 8 * g < kv) ? 1u << ks : 0u;
    }
    if constexpr (!CASE_B) {
      if (XL != 3 || inside) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const uint16_t* base = ubase + opaque_lane(live ? loff[mt] : 0);
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) {
            if constexpr (XL == 3) __builtin_memcpy(&b.x[mt][ks], __builtin_assume_aligned(base + 32 * ks, 2), 16);
            else b.x[mt][ks] = *reinterpret_cast<const uint32x4*>(((b.okm >> ks) & 1u) ? base + 32 * ks : X);
          }
        }
      } else {
        const int top = live ? kv - 1 - b.kb * KB - 8 * gl : 0;  // past the window's end: its last element
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const uint16_t* base = ubase + opaque_lane(live ? loff[mt] : 0);
#pragma unroll
          for (int e = 0; e < 8; e += 2)
            b.x[mt][0][e / 2] = (uint32_t)base[min(e, top)] | (uint32_t)base[min(e + 1, top)] << 16;
        }
      }
    } else {
      const uint16_t* base = ubase + opaque_lane(live ? loff[0] : 0);
      const i64 stride = live ? a.I : 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint16_t* p = base + e * stride;
        uint32x2 v;
        if constexpr (XL == 3) {
          if (inside) {
            __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), 8);
          } else {
            const uint16_t* q = live && b.kb * KB + 8 * g + e < kv ? p : X;
            const i64 room = X + a.total - q;  // at least 1
            uint32_t h[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) h[m] = q[m < room ? m : 0];
            v = uint32x2{h[0] | h[1] << 16, h[2] | h[3] << 16};
          }
        } else {
          v = *reinterpret_cast<const uint32x2*>(p);
        }
        b.x[e / 2][0][2 * (e % 2)] = v[0];
        b.x[e / 2][0][2 * (e % 2) + 1] = v[1];
      }
    }
    if (t + 1 < T) cur.step(a);
  };

  MinNonzero xmin;  // of the lane's X
  // eight j of each of the lane's rows, zero past the window's end
  auto rows_of = [&](const Buf& b, int ks, uint32x4 (&xw)[MT]) {
    if constexpr (!CASE_B) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        xw[mt] = b.x[mt][ks];
        if constexpr (XL == 1) {
          if (!((b.okm >> ks) & 1u)) xw[mt] = uint32x4{};
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        uint32x2 j0 = {b.x[e / 2][0][0], b.x[e / 2][0][1]}, j1 = {b.x[e / 2][0][2], b.x[e / 2][0][3]};
        if constexpr (XL == 3) {
          j0 = __builtin_bit_cast(uint32x2, __builtin_bit_cast(uint64_t, j0) >> shift);
          j1 = __builtin_bit_cast(uint32x2, __builtin_bit_cast(uint64_t, j1) >> shift);
        }
        // low halves of (j0, j1), then high halves
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          xw[2 * h][e / 2] = __builtin_amdgcn_perm(j1[h], j0[h], 0x05040100u);
          xw[2 * h + 1][e / 2] = __builtin_amdgcn_perm(j1[h], j0[h], 0x07060302u);
        }
      }
    }
    if constexpr (XL == 3) {
      if (b.kb * KB + KB > kv) {  // the window's partly filled last block
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const int k = b.kb * KB + 8 * g + e;
          const uint32_t mask = (k < kv ? 0xffffu : 0u) | (k + 1 < kv ? 0xffff0000u : 0u);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) xw[mt][e / 2] &= mask;
        }
      }
    }
  };
  auto compute = [&](int t, const Buf& b) {
    if (t >= T) return;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint32x4 xw[MT];
      rows_of(b, ks, xw);
      if constexpr (EXACT)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int q = 0; q < 4; ++q) xmin.add(xw[mt][q]);
      bf16x8 xv[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xv[mt] = __builtin_bit_cast(bf16x8, xw[mt]);
      // at least four accumulators between two products of one (no MFMA waits
      // for the one just issued), smallest term first
      constexpr int NG = NT >= 2 && !CASE_B ? 2 : 1;
#pragma unroll
      for (int n0 = 0; n0 < NT; n0 += NG) {
        bf16x8 bh[NG], bl[NG], bl2[NG];
#pragma unroll
        for (int u = 0; u < NG; ++u) {
          const int off = (16 * (n0 + u) + c) * PITCH + b.kb * KB + 32 * ks + 8 * g;
          bh[u] = *reinterpret_cast<const bf16x8*>(&sHi[off]);
          bl[u] = *reinterpret_cast<const bf16x8*>(&sLo[off]);
          if constexpr (EXACT) bl2[u] = *reinterpret_cast<const bf16x8*>(&sLo2[off]);
        }
#define TENRSO_BF16_TERM(XB)                                                                       \
  _Pragma("unroll") for (int u = 0; u < NG; ++u) _Pragma("unroll") for (int mt = 0; mt < MT; ++mt) \
      Tacc[mt][n0 + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xv[mt], XB[u], Tacc[mt][n0 + u], 0, 0, 0);
        if constexpr (EXACT) {
          TENRSO_BF16_TERM(bl2)
          TENRSO_BF16_TERM(bl)
          TENRSO_BF16_TERM(bh)
        } else {
          TENRSO_BF16_TERM(bh)
          TENRSO_BF16_TERM(bl)
        }
#undef TENRSO_BF16_TERM
      }
    }
    // a slow index ends, or this wave's range does (it may end inside one)
    if (b.kb == nkb - 1 || t == T - 1) fold_slow<MT, NT>(acc, Tacc, b.pre);
  };

  Buf b[NBUF];
#pragma unroll
  for (int i = 0; i < NBUF - 1; ++i) load(i, b[i]);
  if constexpr (XL > 0) window_zero_tail(fw, kv);
  if constexpr (EXACT) {
    const float fw_min = window_min(fw);
    if (lane == 0) wmin[wave] = fw_min;
    stage_window_store_bf16x3<RT, PITCH, NTH, KWMAX>(sHi, sLo, sLo2, fw);
  } else {
    stage_window_store_bf16x2<RT, PITCH, NTH, KWMAX>(sHi, sLo, fw);
  }
  __syncthreads();  // LDS window staged
  for (int t = 0; t < T; t += NBUF) {
#pragma unroll
    for (int i = 0; i < NBUF; ++i) {
      load(t + i + NBUF - 1, b[(i + NBUF - 1) % NBUF]);
      compute(t + i, b[i]);
    }
  }

  float* out = partial + (i64)split * a.I * a.R;
  if constexpr (EXACT) {
    // not finite, or too small for exact parts of FAST or for T (the bounds of the fp32
    // kernel): all of it again in fp32
    const float xm = xmin.value();  // of the lane
    float fm = wmin[0];
#pragma unroll
    for (int v = 1; v < WAVES; ++v) fm = fminf(fm, wmin[v]);
    const bool small = fm < 0x1p-108f || xm * fm < 0x1p-123f;
    if (__any(small || !(sum_of_zeros<MT, NT>(acc) == 0.f))) redo = 1;
    __syncthreads();
    if (redo) {
      redo_window<RT, NTH, KWMAX>(smem, a, w, kv);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = floatx4{0.f, 0.f, 0.f, 0.f};
      cur = BlockCursor<KB, CASE_B>(a, s_lo + wq, w, nkb, wr);
      __syncthreads();
#pragma unroll 1
      for (int t = 0; t < T; ++t) {
        load(t, b[0]);
        uint32x4 xw[MT];
        rows_of(b[0], 0, xw);
        floatx8 x[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int e = 0; e < 8; ++e)
            x[mt][e] = __uint_as_float(e % 2 ? xw[mt][e / 2] & 0xffff0000u : xw[mt][e / 2] << 16);
        redo_block(acc, x, b[0].pre, smem, c, b[0].kb * KB + 8 * g, kv);
      }
      __syncthreads();  // window no longer read
    }
  }
  wg_reduce_store<MT, NT, WAVES, !EXACT>(acc, smem, wave, lane, out, a.I, a.R, a.r0, a.rcount, row_base, CASE_B);
}

// ---------------------------------------------------------------------------
// What the MFMA kernels do not take: empty contractions (the result is zero) and a
// tensor that is not aligned to its own element type.  One thread per (i, r); grid.y
// splits j.
// ---------------------------------------------------------------------------
struct GenericArgs {
  int nd, mode, n_oth;
  i64 I, Q, R, J;
  i64 oth_size[MAXD];
  const float* oth_fac[MAXD];
  int splits;
  int bf16;
};

__global__ __launch_bounds__(256) void mttkrp_generic(const void* __restrict__ Xv, GenericArgs a,
                                                      float* __restrict__ partial) {
  const i64 idx = (i64)blockIdx.x * 256 + threadIdx.x;
  if (idx >= a.I * a.R) return;
  const i64 i = idx / a.R, r = idx - (idx / a.R) * a.R;
  const int split = blockIdx.y;
  const i64 j_begin = (i64)split * a.J / a.splits, j_end = (i64)(split + 1) * a.J / a.splits;
  float acc = 0.f;
  for (i64 j = j_begin; j < j_end; ++j) {
    i64 rem = j;
    float kr = 1.f;
    for (int m = a.n_oth - 1; m >= 0; --m) {
      const i64 sz = a.oth_size[m];
      const i64 ix = rem % sz;
      rem /= sz;
      kr *= a.oth_fac[m][ix * a.R + r];
    }
    const i64 p = j / a.Q, q = j - p * a.Q;
    const i64 off = (p * a.I + i) * a.Q + q;
    float x;
    if (a.bf16) {
      const uint16_t h = reinterpret_cast<const uint16_t*>(Xv)[off];
      x = __uint_as_float((uint32_t)h << 16);
    } else {
      x = reinterpret_cast<const float*>(Xv)[off];
    }
    acc = fmaf(x, kr, acc);
  }
  partial[(i64)split * a.I * a.R + idx] = acc;
}

// ---------------------------------------------------------------------------
// Reduction of split partials (fixed order, FP64) and conversions.
// ---------------------------------------------------------------------------
// A workgroup owns 64 consecutive outputs and splits the split range into
// RED_GROUPS contiguous pieces, one per group of 64 threads (each lane one
// output, so every load of a group is one contiguous 256-byte row segment).
// Each group sums its piece in FP64 with four independent chains; the group
// sums are then added in group order.  The order is fixed, so the result is
// run-to-run identical.  (One thread per output looping over all splits left
// 12 workgroups for a 96^4 rank-32 result, a latency chain of ~170 loads.)
constexpr int RED_GROUPS = 16;
__device__ __forceinline__ void reduce_partials_body(const float* __restrict__ part, int splits, i64 n, i64 block,
                                                     float* __restrict__ o32, double* __restrict__ o64) {
  __shared__ double red[RED_GROUPS][64];
  const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6;
  const i64 idx = block * 64 + lane;
  double s = 0.0;
  if (idx < n) {
    const int s0 = (int)((i64)grp * splits / RED_GROUPS), s1 = (int)((i64)(grp + 1) * splits / RED_GROUPS);
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    int sp = s0;
    for (; sp + 4 <= s1; sp += 4) {
      a0 += (double)part[(i64)(sp + 0) * n + idx];
      a1 += (double)part[(i64)(sp + 1) * n + idx];
      a2 += (double)part[(i64)(sp + 2) * n + idx];
      a3 += (double)part[(i64)(sp + 3) * n + idx];
    }
    for (; sp < s1; ++sp) a0 += (double)part[(i64)sp * n + idx];
    s = (a0 + a1) + (a2 + a3);
  }
  red[grp][lane] = s;
  __syncthreads();
  if (grp == 0 && idx < n) {
    double t = red[0][lane];
#pragma unroll
    for (int g = 1; g < RED_GROUPS; ++g) t += red[g][lane];
    if (o32) o32[idx] = (float)t;
    if (o64) o64[idx] = t;
  }
}
__global__ __launch_bounds__(64 * RED_GROUPS) void reduce_partials_kernel(const float* __restrict__ part, int splits,
                                                                          i64 n, float* __restrict__ o32,
                                                                          double* __restrict__ o64) {
  reduce_partials_body(part, splits, n, blockIdx.x, o32, o64);
}
// The partials of several MTTKRPs in one launch: result m takes the workgroups
// [first[m], first[m + 1]).
struct ReduceMany {
  int count;
  const float* part[MAXD];
  int splits[MAXD];
  i64 n[MAXD];
  float* out[MAXD];
  unsigned first[MAXD + 1];
};
__global__ __launch_bounds__(64 * RED_GROUPS) void reduce_many_kernel(ReduceMany r) {
  int m = 0;
  while (m + 1 < r.count && blockIdx.x >= r.first[m + 1]) ++m;
  reduce_partials_body(r.part[m], r.splits[m], r.n[m], blockIdx.x - r.first[m], r.out[m], nullptr);
}

// vec: src 16-byte and dst 8-byte aligned (checked on the host), else scalar
__global__ __launch_bounds__(256) void f32_to_bf16_kernel(const float* __restrict__ src, i64 n,
                                                          uint16_t* __restrict__ dst, int vec) {
  const i64 i4 = ((i64)blockIdx.x * 256 + threadIdx.x) * 4;
  if (vec && i4 + 3 < n) {
    const floatx4 v = *reinterpret_cast<const floatx4*>(src + i4);
    ushort4 o;
    o.x = f32_to_bf16_rne(v[0]);
    o.y = f32_to_bf16_rne(v[1]);
    o.z = f32_to_bf16_rne(v[2]);
    o.w = f32_to_bf16_rne(v[3]);
    *reinterpret_cast<ushort4*>(dst + i4) = o;
  } else {
    for (i64 i = i4; i < n; ++i) dst[i] = f32_to_bf16_rne(src[i]);
  }
}

// [rows, K] -> [K, rows] transpose through a 32x32 LDS tile.
// With B < Bp the output rows are padded: input row r = a*B + b lands at
// a*Bp + b of an output row of extent (rows / B) * Bp (the pad entries are
// zero-filled beforehand); B = Bp leaves the layout plain.
__global__ __launch_bounds__(256) void transpose_kernel(const float* __restrict__ src, i64 rows, i64 K,
                                                        float* __restrict__ dst, i64 B = 1, i64 Bp = 1) {
  __shared__ float tile[32][33];
  const i64 r0 = (i64)blockIdx.y * 32, k0 = (i64)blockIdx.x * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int yy = ty; yy < 32; yy += 8) {
    const i64 r = r0 + yy, k = k0 + tx;
    tile[yy][tx] = (r < rows && k < K) ? src[r * K + k] : 0.f;
  }
  __syncthreads();
  for (int yy = ty; yy < 32; yy += 8) {
    const i64 k = k0 + yy, r = r0 + tx;
    if (k < K && r < rows) {
      const i64 o = B == Bp ? k * rows + r : k * (rows / B * Bp) + (r / B) * Bp + r % B;
      dst[o] = tile[tx][yy];
    }
  }
}

// Forward-order Khatri-Rao of n factors: row = (i_0, ..., i_{n-1}) last fastest.
struct KrManyArgs {
  int n;
  i64 R, rows;
  i64 sizes[MAXD];
  const float* F[MAXD];
};
__device__ __forceinline__ void kr_many_body(const KrManyArgs& a, float* __restrict__ dst) {
  const i64 idx = (i64)blockIdx.x * 256 + threadIdx.x;
  if (idx >= a.rows * a.R) return;
  const i64 row = idx / a.R, r = idx - (idx / a.R) * a.R;
  i64 rem = row;
  float v = 1.f;
  float vals[MAXD];
  for (int m = a.n - 1; m >= 0; --m) {
    const i64 ix = rem % a.sizes[m];
    rem /= a.sizes[m];
    vals[m] = a.F[m][ix * a.R + r];
  }
  for (int m = 0; m < a.n; ++m) v = v * vals[m];  // left-to-right, as khatri_rao_except_mode
  dst[idx] = v;
}
__global__ __launch_bounds__(256) void kr_many_kernel(KrManyArgs a, float* __restrict__ dst) { kr_many_body(a, dst); }

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static inline unsigned cdiv(i64 a, i64 b) { return (unsigned)((a + b - 1) / b); }

int reduce_partials(tenrso_ctx* ctx, const float* partial, int splits, i64 n, float* out32, double* out64) {
  if (n == 0) return TENRSO_OK;
  hipLaunchKernelGGL(reduce_partials_kernel, dim3(cdiv(n, 64)), dim3(64 * RED_GROUPS), 0, ctx->stream, partial,
                     splits, n, out32, out64);
  TENRSO_HIP_TRY(hipGetLastError());
  return TENRSO_OK;
}

// Several Khatri-Rao products in one launch: product y of grid.y into dst[y].
constexpr int KR_BATCH = MAXD;
struct KrBatchArgs {
  int count;
  KrManyArgs k[KR_BATCH];
  float* dst[KR_BATCH];
};
__global__ __launch_bounds__(256) void kr_batch_kernel(KrBatchArgs b) {
  const int y = blockIdx.y;
  if (y >= b.count) return;
  kr_many_body(b.k[y], b.dst[y]);
}

int mttkrp_pre_batch(tenrso_ctx* ctx, int nd, const i64* shape, const float* const* F, i64 R, int nmodes,
                     const int* modes, bool via_copy_last, const float** pre) {
  KrBatchArgs b{};
  int owner[KR_BATCH];  // the product each requested mode uses, or -1
  i64 offs[KR_BATCH + 1] = {0};
  for (int i = 0; i < nmodes; ++i) {
    pre[i] = nullptr;
    owner[i] = -1;
    const int mode = modes[i];
    // the PRE factors: every other mode but the fastest, in order (the last
    // mode through the copy contracts modes 0 .. nd-3 the same way)
    KrManyArgs k{};
    k.R = R;
    k.rows = 1;
    const bool copy = via_copy_last && mode == nd - 1;
    const int n_oth = nd - 1;
    if (n_oth < 3) continue;
    for (int j = 0; j < nd && k.n < n_oth - 1; ++j) {
      if (!copy && j == mode) continue;
      k.F[k.n] = F[j];
      k.sizes[k.n] = shape[j];
      k.rows *= shape[j];
      ++k.n;
    }
    // shared with an earlier product of the same factors?
    for (int q = 0; q < b.count && owner[i] < 0; ++q) {
      bool same = b.k[q].n == k.n;
      for (int j = 0; same && j < k.n; ++j) same = b.k[q].F[j] == k.F[j] && b.k[q].sizes[j] == k.sizes[j];
      if (same) owner[i] = q;
    }
    if (owner[i] < 0) {
      if (b.count == KR_BATCH) continue;  // more distinct products than one launch takes: the MTTKRP forms its own
      owner[i] = b.count;
      b.k[b.count] = k;
      offs[b.count + 1] = offs[b.count] + k.rows * R;
      ++b.count;
    }
  }
  if (b.count == 0) return TENRSO_OK;
  void* buf = nullptr;
  TENRSO_TRY(ctx_buffer(ctx, SLOT_PRE, (size_t)offs[b.count] * sizeof(float), &buf));
  i64 maxn = 0;
  for (int q = 0; q < b.count; ++q) {
    b.dst[q] = (float*)buf + offs[q];
    maxn = std::max(maxn, b.k[q].rows * R);
  }
  for (int i = 0; i < nmodes; ++i)
    if (owner[i] >= 0) pre[i] = b.dst[owner[i]];
  hipLaunchKernelGGL(kr_batch_kernel, dim3(cdiv(maxn, 256), b.count), dim3(256), 0, ctx->stream, b);
  TENRSO_HIP_TRY(hipGetLastError());
  return TENRSO_OK;
}

int khatri_rao_many(tenrso_ctx* ctx, int n, const float* const* F, const i64* sizes, i64 R, float* dst) {
  KrManyArgs a{};
  a.n = n;
  a.R = R;
  a.rows = 1;
  for (int m = 0; m < n; ++m) {
    a.sizes[m] = sizes[m];
    a.F[m] = F[m];
    a.rows *= sizes[m];
  }
  hipLaunchKernelGGL(kr_many_kernel, dim3(cdiv(a.rows * R, 256)), dim3(256), 0, ctx->stream, a, dst);
  TENRSO_HIP_TRY(hipGetLastError());
  return TENRSO_OK;
}

int convert_bf16(tenrso_ctx* ctx, const float* src, i64 n, uint16_t* dst) {
  if (n == 0) return TENRSO_OK;
  const int vec = (uintptr_t)src % 16 == 0 && (uintptr_t)dst % 8 == 0;
  hipLaunchKernelGGL(f32_to_bf16_kernel, dim3(cdiv(cdiv(n, 4), 256)), dim3(256), 0, ctx->stream, src, n, dst, vec);
  TENRSO_HIP_TRY(hipGetLastError());
  return TENRSO_OK;
}

// [rows, K] fp32 -> [rows, Kp] bf16 (RNE), zero in the pad columns k >= K
// one workgroup per row (no division per element)
__global__ __launch_bounds__(256) void f32_to_bf16_pad_kernel(const float* __restrict__ src, i64 K, i64 Kp,
                                                              uint16_t* __restrict__ dst) {
  const i64 r = blockIdx.x;
  for (i64 k = threadIdx.x; k < Kp; k += 256) dst[r * Kp + k] = k < K ? f32_to_bf16_rne(src[r * K + k]) : (uint16_t)0;
}

int convert_bf16_padded(tenrso_ctx* ctx, const float* src, int nd, const i64* shape, i64 Kp, uint16_t* dst) {
  i64 total = 1;
  for (int k = 0; k < nd; ++k) total *= shape[k];
  const i64 K = shape[nd - 1];
  if (total == 0) return TENRSO_OK;
  const i64 rows = total / K;
  hipLaunchKernelGGL(f32_to_bf16_pad_kernel, dim3((unsigned)rows), dim3(256), 0, ctx->stream, src, K, Kp, dst);
  TENRSO_HIP_TRY(hipGetLastError());
  return TENRSO_OK;
}

// one workgroup per row (no division per element)
__global__ __launch_bounds__(256) void f32_pad_kernel(const float* __restrict__ src, i64 K, i64 Kp,
                                                      float* __restrict__ dst) {
  const i64 r = blockIdx.x;
  for (i64 k = threadIdx.x; k < Kp; k += 256) dst[r * Kp + k] = k < K ? src[r * K + k] : 0.0f;
}

// zeros at [B, Bp) of each of n rows of Bp (the pads of a padded copy, nothing else)
__global__ __launch_bounds__(256) void zero_pads_kernel(float* __restrict__ dst, i64 n, i64 B, i64 Bp) {
  const i64 np = Bp - B;
  const i64 e = (i64)blockIdx.x * 256 + threadIdx.x;
  if (e >= n * np) return;
  const i64 r = e / np;
  dst[r * Bp + B + (e - r * np)] = 0.0f;
}

int copy_f32_padded(tenrso_ctx* ctx, const float* src, int nd, const i64* shape, i64 Kp, float* dst) {
  i64 total = 1;
  for (int k = 0; k < nd; ++k) total *= shape[k];
  const i64 K = shape[nd - 1];
  if (total == 0) return TENRSO_OK;
  const i64 rows = total / K;
  hipLaunchKernelGGL(f32_pad_kernel, dim3((unsigned)rows), dim3(256), 0, ctx->stream, src, K, Kp, dst);
  TENRSO_HIP_TRY(hipGetLastError());
  return TENRSO_OK;
}

int transpose_last_to_front_f32_padded(tenrso_ctx* ctx, const float* src, int nd, const i64* shape, i64 Bp,
                                       float* dst) {
  i64 total = 1;
  for (int k = 0; k < nd; ++k) total *= shape[k];
  if (total == 0) return TENRSO_OK;
  const i64 K = shape[nd - 1], rows = total / K, B = shape[nd - 2];
  const i64 nrow = K * (rows / B);  // rows of Bp in the copy
  if (Bp != B)
    hipLaunchKernelGGL(zero_pads_kernel, dim3(cdiv(nrow * (Bp - B), 256)), dim3(256), 0, ctx->stream, dst, nrow, B,
                       Bp);
  hipLaunchKernelGGL(transpose_kernel, dim3(cdiv(K, 32), cdiv(rows, 32)), dim3(256), 0, ctx->stream,
                     src, rows, K, dst, B, Bp);
  TENRSO_HIP_TRY(hipGetLastError());
  return TENRSO_OK;
}

int transpose_last_to_front_f32(tenrso_ctx* ctx, const float* src, int nd, const i64* shape, float* dst) {
  i64 total = 1;
  for (int k = 0; k < nd; ++k) total *= shape[k];
  if (total == 0) return TENRSO_OK;
  const i64 K = shape[nd - 1], rows = total / K;
  hipLaunchKernelGGL(transpose_kernel, dim3(cdiv(K, 32), cdiv(rows, 32)), dim3(256), 0, ctx->stream,
                     src, rows, K, dst);
  TENRSO_HIP_TRY(hipGetLastError());
  return TENRSO_OK;
}

// bf16 copy of an fp32 tensor (RNE, as f32_to_bf16_kernel) and per-workgroup (sum of
// squares, min) partials in one pass: 16-byte loads, grid-stride.
__global__ __launch_bounds__(256) void convert_bf16_norm_kernel(const float* __restrict__ X, i64 n4,
                                                                uint16_t* __restrict__ dst,
                                                                double* __restrict__ part) {
  __shared__ double red[256];
  const int tid = threadIdx.x;
  const floatx4* X4 = reinterpret_cast<const floatx4*>(X);
  ushort4* d4 = reinterpret_cast<ushort4*>(dst);
  const i64 stride = (i64)gridDim.x * 256;
  double ss = 0.0;
  float mn = FLT_MAX;
  auto one = [&](i64 i, const floatx4& v) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      ss = fma((double)v[q], (double)v[q], ss);
      mn = fminf(mn, v[q]);
    }
    ushort4 o;
    o.x = f32_to_bf16_rne(v[0]);
    o.y = f32_to_bf16_rne(v[1]);
    o.z = f32_to_bf16_rne(v[2]);
    o.w = f32_to_bf16_rne(v[3]);
    d4[i] = o;
  };
  i64 i = (i64)blockIdx.x * 256 + tid;
  for (; i + 3 * stride < n4; i += 4 * stride) {
    floatx4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = X4[i + u * stride];
#pragma unroll
    for (int u = 0; u < 4; ++u) one(i + u * stride, v[u]);
  }
  for (; i < n4; i += stride) one(i, X4[i]);
  // (sum, min) partial of the workgroup
  double v = ss;
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if ((tid & 63) == 0) red[tid >> 6] = v;
  __syncthreads();
  const double tot = (red[0] + red[1]) + (red[2] + red[3]);
  __syncthreads();
  red[tid] = (double)mn;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (tid < k) red[tid] = fmin(red[tid], red[tid + k]);
    __syncthreads();
  }
  if (tid == 0) {
    part[blockIdx.x] = tot;
    part[gridDim.x + blockIdx.x] = red[0];
  }
}

int convert_bf16_norm(tenrso_ctx* ctx, const float* X, i64 total, uint16_t* dst, double* tmp, int* nblk_out) {
  *nblk_out = 0;
  if (total == 0 || total % 4 != 0 || (uintptr_t)X % 16 != 0) return TENRSO_ERR_UNSUPPORTED;
  const int nblk = (int)std::min<i64>(1024, cdiv(total / 4, 256 * 4));
  hipLaunchKernelGGL(convert_bf16_norm_kernel, dim3(nblk), dim3(256), 0, ctx->stream, X, total / 4, dst, tmp);
  TENRSO_HIP_TRY(hipGetLastError());
  *nblk_out = nblk;
  return TENRSO_OK;
}

namespace {

// The bf16 instance for nt rank tiles of 16, blocks of 32 ks elements, wv (16-byte
// window loads) and the load form xl.  ks = 2 only in case A with xl 0 (a fastest
// mode divisible by 64 is never ragged).
constexpr int BF16_WAVES = 8, BF16_KWMAX = 128;
template <int NT, bool CASE_B, bool WV>
const void* bf16_pick(int ks, int xl) {
  constexpr int W = BF16_WAVES, K = BF16_KWMAX;
  if constexpr (!CASE_B) {
    if (ks == 2) return reinterpret_cast<const void*>(mttkrp_bf16_mfma<NT, W, 2, K, CASE_B, WV, 0>);
    if (xl == 4) return reinterpret_cast<const void*>(mttkrp_bf16_mfma<NT, W, 1, K, CASE_B, WV, 4>);
  }
  if (xl == 0) return reinterpret_cast<const void*>(mttkrp_bf16_mfma<NT, W, 1, K, CASE_B, WV, 0>);
  if constexpr (!CASE_B) {
    if (xl == 1) return reinterpret_cast<const void*>(mttkrp_bf16_mfma<NT, W, 1, K, CASE_B, WV, 1>);
  }
  return reinterpret_cast<const void*>(mttkrp_bf16_mfma<NT, W, 1, K, CASE_B, WV, 3>);
}
template <int NT>
const void* bf16_pick(bool case_b, bool wv, int ks, int xl) {
  if (case_b) return wv ? bf16_pick<NT, true, true>(ks, xl) : bf16_pick<NT, true, false>(ks, xl);
  return wv ? bf16_pick<NT, false, true>(ks, xl) : bf16_pick<NT, false, false>(ks, xl);
}
const void* mttkrp_bf16_kernel(int nt, bool case_b, bool wv, int ks, int xl) {
  return nt == 1 ? bf16_pick<1>(case_b, wv, ks, xl)
                 : (nt == 2 ? bf16_pick<2>(case_b, wv, ks, xl) : bf16_pick<4>(case_b, wv, ks, xl));
}

struct Plan {
  i64 P = 1, I = 1, Q = 1, J = 1;
  int n_oth = 0;
  int oth[MAXD];
  i64 oth_size[MAXD];
  i64 fast_size = 1;
};

Plan make_plan(int nd, const i64* shape, int mode) {
  Plan p;
  for (int k = 0; k < mode; ++k) p.P *= shape[k];
  for (int k = mode + 1; k < nd; ++k) p.Q *= shape[k];
  p.I = shape[mode];
  p.J = p.P * p.Q;
  for (int k = 0; k < nd; ++k)
    if (k != mode) {
      p.oth[p.n_oth] = k;
      p.oth_size[p.n_oth] = shape[k];
      ++p.n_oth;
    }
  p.fast_size = p.n_oth ? p.oth_size[p.n_oth - 1] : 1;
  return p;
}

}  // namespace

// How a mode runs in the fp32 MFMA kernel (ok: it can, in one launch of up to 64 rank
// columns); its splits are still to be chosen.
struct X3Plan {
  bool ok = false, case_b = false;
  int nt = 0, xl = 0;
  KernArgs a;
};

// resident workgroups of a kernel on one CU (occupancy query, cached)
static int occupancy(tenrso_ctx* ctx, const void* kern, int threads, int* occ) {
  for (int i = 0; i < ctx->occ_n; ++i)
    if (ctx->occ_kern[i] == kern) {
      *occ = ctx->occ_val[i];
      return TENRSO_OK;
    }
  int nb = 0;
  TENRSO_HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kern, threads, 0));
  *occ = std::max(1, nb);
  if (ctx->occ_n < (int)(sizeof(ctx->occ_val) / sizeof(ctx->occ_val[0]))) {
    ctx->occ_kern[ctx->occ_n] = kern;
    ctx->occ_val[ctx->occ_n++] = *occ;
  }
  return TENRSO_OK;
}

constexpr i64 MAX_THREADS = UINT32_MAX;  // of a launch in one dimension

// a.slow_splits splits of the slow range, balanced
static void set_splits(KernArgs& a, i64 ssp) {
  a.slow_splits = (int)std::max<i64>(1, ssp);
  a.slow_q = a.n_slow / a.slow_splits;
  a.slow_rem = a.n_slow % a.slow_splits;
}

int mttkrp_dense(tenrso_ctx* ctx, int prec, const void* X, const void* X_t, int nd, const i64* shape,
                 const float* const* F, i64 R, int mode, MttkrpOut outk, void* out, MttkrpResult* res,
                 const AlsJob* job, const MttkrpScratch* scratch, i64 x_pad, i64 xt_pad,
                 const float* pre_rows, bool want_norm, int slot, X3Plan* plan) {
  Plan pl = make_plan(nd, shape, mode);
  const bool bf16 = prec == TENRSO_PREC_BF16;
  const float* Fv[MAXD];
  for (int k = 0; k < nd; ++k) Fv[k] = F[k];
  const void* Xuse = X;
  int mode_use = mode;
  i64 shape_use[MAXD];
  for (int k = 0; k < nd; ++k) shape_use[k] = shape[k];

  // With a last-to-front copy given (fp32, also of a BF16 call), the last mode runs
  // as mode 0 of the copy (same j order).
  bool x3 = false;
  if (X_t && mode == nd - 1 && nd >= 2) {
    x3 = bf16;
    Xuse = X_t;
    mode_use = 0;
    shape_use[0] = shape[nd - 1];
    Fv[0] = F[nd - 1];
    for (int k = 1; k < nd; ++k) {
      shape_use[k] = shape[k - 1];
      Fv[k] = F[k - 1];
    }
    pl = make_plan(nd, shape_use, 0);
  }

  const i64 I = pl.I;
  const i64 nout = I * R;
  // rank columns of a launch: up to 64, or 128 of an fp32 tensor (for ranks 65 to 128
  // one pass over X, which can carry the wide-rank job: an ALS mode at 256^3 rank 128
  // takes 48 us so, against two launches of 25 us beside the job on a side stream and
  // about 28 us of waits between the streams)
  const int RT = R <= 16 ? 16 : (R <= 32 ? 32 : (R <= 64 || (bf16 && !x3) ? 64 : 128));
  const int NT = RT / 16;
  const int rchunks = (int)((R + RT - 1) / RT);

  // PRE: product of the other modes except the fastest (forward order).
  const float* pre = nullptr;
  size_t scratch_used = 0;  // bytes of the caller's workspace taken by PRE
  // the most split partials that fit in the caller's workspace (or no bound)
  auto max_splits = [&]() -> i64 {
    if (!scratch) return INT64_MAX;
    const size_t per = (size_t)std::max<i64>(1, nout) * sizeof(float);
    return scratch->bytes > scratch_used ? (i64)((scratch->bytes - scratch_used) / per) : 0;
  };
  auto partial_buffer = [&](int nsplits, float** p) -> int {
    if (scratch) {
      *p = reinterpret_cast<float*>(static_cast<char*>(scratch->base) + scratch_used);
      return TENRSO_OK;
    }
    void* pbuf = nullptr;
    TENRSO_TRY(ctx_buffer(ctx, slot, (size_t)nsplits * nout * sizeof(float), &pbuf));
    *p = (float*)pbuf;
    return TENRSO_OK;
  };
  auto too_small = [&](i64 need_splits) {
    set_error("workspace of %zu bytes is too small for this MTTKRP (needs %zu bytes)", scratch->bytes,
              scratch_used + (size_t)need_splits * (size_t)std::max<i64>(1, nout) * sizeof(float));
    return TENRSO_ERR_UNSUPPORTED;
  };
  if (pl.n_oth >= 3 && pre_rows) {
    pre = pre_rows;
  } else if (pl.n_oth >= 3) {
    const float* pf[MAXD];
    i64 ps[MAXD];
    i64 prows = 1;
    for (int m = 0; m < pl.n_oth - 1; ++m) {
      pf[m] = Fv[pl.oth[m]];
      ps[m] = pl.oth_size[m];
      prows *= ps[m];
    }
    void* buf = nullptr;
    const size_t pre_bytes = (size_t)(prows * R) * sizeof(float);
    if (scratch) {
      if (pre_bytes > scratch->bytes) {
        set_error("workspace of %zu bytes cannot hold the %zu bytes of Khatri-Rao rows", scratch->bytes, pre_bytes);
        return TENRSO_ERR_UNSUPPORTED;
      }
      buf = scratch->base;
      scratch_used = (pre_bytes + 255) / 256 * 256;
    } else {
      TENRSO_TRY(ctx_buffer(ctx, SLOT_TMP, pre_bytes, &buf));
    }
    TENRSO_TRY(khatri_rao_many(ctx, pl.n_oth - 1, pf, ps, R, (float*)buf));
    pre = (const float*)buf;
  } else if (pl.n_oth == 2) {
    pre = Fv[pl.oth[0]];
  }
  const float* fastf = pl.n_oth ? Fv[pl.oth[pl.n_oth - 1]] : nullptr;

  // a last mode of one row is a contiguous vector of j: case A with Q = J
  const bool caseB = pl.Q == 1 && pl.I != 1;
  // memory extent of the fastest other mode: the BF16 ALS copies of a tensor
  // whose last mode is no multiple of the load vector have that mode padded
  // (zeros), so every row starts on a vector boundary
  const i64 pad = mode == nd - 1 && nd >= 2 ? xt_pad : x_pad;
  const i64 fast_stride = (pad > 0 && !caseB) ? pad : pl.fast_size;
  const i64 Qcon = !caseB && pl.Q == 1 ? pl.J : pl.Q;
  const i64 Qmem = (pad > 0 && !caseB) ? Qcon / pl.fast_size * pad : Qcon;

  KernArgs a{};
  a.I = I;
  a.Q = Qmem;
  a.R = R;
  a.fast_size = pl.fast_size;
  a.fast_stride = fast_stride;
  a.pre = pre;
  a.fast = fastf;

  const bool fp32 = !bf16 || x3;
  const int KB = !fp32 && !caseB && pl.fast_size % 64 == 0 && (uintptr_t)Xuse % 16 == 0 ? 64 : 32;
  constexpr int KWMAX = 128;  // LDS window bound (64 x 136 bf16, three planes)
  // LDS window of the fastest mode: the largest multiple of KB that divides it.
  // A fastest mode no such window divides ("ragged", e.g. 100 or 250) takes
  // windows of a multiple of 32 rows covering it as evenly as possible, the last
  // one partly filled and masked (XL 1).
  int kw = 0;
  for (i64 cand = std::min<i64>(KWMAX, pl.fast_size) / KB * KB; cand >= KB; cand -= KB)
    if (pl.fast_size % cand == 0) {
      kw = (int)cand;
      break;
    }
  const uintptr_t xaddr = (uintptr_t)Xuse;
  int XL = 0;
  if (kw == 0 && pl.fast_size > 0) {
    const i64 nw = (pl.fast_size + KWMAX - 1) / KWMAX;
    kw = (int)(((pl.fast_size + nw - 1) / nw + 31) / 32 * 32);
    XL = 1;
  }
  // Case A on a zero-padded copy whose rows reach a multiple of 32: every
  // window's last block ends inside the padded row, so X loads need no masks
  // (the pads are zero, and window rows past kv are staged as zeros); only the
  // window load keeps kv (XL 4)
  if (!caseB && pad > 0 && XL == 1 && xaddr % 16 == 0 && fast_stride >= (pl.fast_size + 31) / 32 * 32) XL = 4;
  // The unmasked forms read aligned vectors: 16 bytes of a row; in case B 8 bytes of
  // two (fp32) or four (bf16) rows.  Every other tensor, at any alignment of its
  // type, takes XL 1 (fp32) or, unless its rows are 16-byte aligned, XL 3 (bf16).
  if (XL == 0 && (caseB ? I % (fp32 ? 2 : 4) != 0 || xaddr % 8 != 0 : xaddr % 16 != 0)) XL = 1;
  if (!fp32 && XL == 1 && (caseB || fast_stride % 8 != 0 || xaddr % 16 != 0)) XL = 3;
  const bool mfma_ok = pl.n_oth >= 1 && pl.J > 0 && kw > 0 && I > 0 && xaddr % (fp32 ? 4 : 2) == 0;

  float* partial = nullptr;
  int splits = 1;
  const double* norm = nullptr;
  int nnorm = 0;
  if (mfma_ok) {
    const i64 rows_per_wg = !fp32 && caseB ? 64 : 32;
    const i64 rtiles = (i64)cdiv(I, rows_per_wg);
    const i64 tiles = rtiles * rchunks;
    a.kw = kw;
    a.nwin = (int)((pl.fast_size + kw - 1) / kw);
    a.n_slow = pl.J / pl.fast_size;
    a.qs = caseB ? 1 : Qmem / fast_stride;
    a.total = caseB ? pl.J * I : pl.J / Qcon * I * Qmem;
    a.rtiles = (int)rtiles;
    a.win_vec = (R % 4 == 0) && ((uintptr_t)fastf % 16 == 0);
    if (plan) {
      plan->ok = fp32 && NT < 8 && rchunks == 1;
      plan->a = a;
      plan->a.rcount = (int)R;
      plan->case_b = caseB;
      plan->nt = NT;
      plan->xl = XL;
      return TENRSO_OK;
    }
    // 8-wave workgroups, one per CU (the register budget admits one), so a fused
    // ALS job gets a CU of its own instead of sharing one with an MTTKRP workgroup
    // (measured: the job at ~22 us beside the MTTKRP against ~14 us alone).  When
    // the job shares the launch it takes one of the resident slots, so every
    // workgroup is resident at once.
    int waves = 8, occ = 0;
    const void* kern = !fp32 ? mttkrp_bf16_kernel(NT, caseB, a.win_vec, KB / 32, XL)
                             : (NT == 8 ? mttkrp_x3_kernel_n8(caseB, a.win_vec, XL)
                                        : mttkrp_x3_kernel_w8(NT, caseB, a.win_vec, XL));
    TENRSO_TRY(occupancy(ctx, kern, waves * 64, &occ));
    int wpc = bf16 ? ctx->wg_per_cu_bf16 : ctx->wg_per_cu_f32;  // TENRSO_WG_PER_CU_* override
    if (wpc <= 0) wpc = std::min(occ, 2);
    const bool fuse_job = job != nullptr && rchunks == 1 && (job->R <= JOB_NE || NT == 8) && (fp32 || !caseB);
    i64 target = (i64)wpc * ctx->num_cus - ((fuse_job && occ <= wpc) ? 1 : 0);
    // Splits of the slow range: the count with the least (rounds of resident
    // workgroups) x (blocks of its slowest wave + 3), a workgroup's start and end
    // costing about three blocks; at least one block a wave where there are as many.
    // At 256^3 rank 64 that is one round (16 splits, 256 workgroups; two rounds of
    // half the work took 25 us against 18).
    const i64 wgs1 = std::max<i64>(1, tiles) * a.nwin, nkb = (kw + KB - 1) / KB;
    const i64 most = std::max<i64>(1, std::min<i64>(a.n_slow * nkb / waves, a.n_slow));
    // The candidates: for every number of rounds the fewest splits with the blocks of
    // the most that it holds.
    i64 ssp = 1, best = INT64_MAX;
    const i64 round0 = (wgs1 + target - 1) / target;
    for (i64 rounds = round0; rounds <= round0 + 8; ++rounds) {
      i64 s = std::min<i64>(most, rounds * target / wgs1);
      if (s < 1) continue;
      const i64 blocks = ((a.n_slow + s - 1) / s * nkb + waves - 1) / waves;
      const i64 per = std::max<i64>(1, blocks * waves / nkb);  // slow indices a workgroup can take in as many
      s = std::min(s, (a.n_slow + per - 1) / per);
      if (rounds * (blocks + 3) < best) {
        best = rounds * (blocks + 3);
        ssp = s;
      }
    }
    // With the job fused a launch of few blocks lasts as long as the job, and fewer
    // splits leave the row solve less to add: one round, and a slow index a wave
    // (224x96x128 rank 5: solve 4.5 us behind 12 splits, 5.1 behind 36).
    if (fuse_job) ssp = std::max<i64>(1, std::min<i64>(target / wgs1, a.n_slow / waves));
    // Several rounds and no job: 4-wave workgroups, as many splits as bring 1.5
    // times the resident ones while a wave keeps four blocks (9216 rows, 9216 j,
    // rank 32: 75 us with 576 workgroups, 70 with 1152, 69 with 1728).
    const bool with_norm = want_norm && fp32 && !bf16 && pad == 0 && !job && rchunks == 1 && NT < 8;
    if (fp32 && NT < 8 && !fuse_job && (wgs1 * ssp > target || with_norm)) {
      kern = with_norm ? mttkrp_x3_kernel_norm(NT, caseB, a.win_vec, XL)
                       : mttkrp_x3_kernel_w4(NT, caseB, a.win_vec, XL);
      waves = 4;
      TENRSO_TRY(occupancy(ctx, kern, waves * 64, &occ));
      target = (i64)(ctx->wg_per_cu_f32 > 0 ? ctx->wg_per_cu_f32 : occ) * ctx->num_cus;
      ssp = std::min<i64>((3 * target / 2 + wgs1 - 1) / wgs1, a.n_slow * nkb / (4 * waves));
      ssp = std::max<i64>(1, std::min<i64>(ssp, a.n_slow));
    }
    ssp = std::min<i64>(ssp, 65535 / a.nwin);
    // a caller's workspace bounds the partials: fewer splits, or refuse
    if (max_splits() < a.nwin) return too_small(a.nwin);
    ssp = std::min<i64>(ssp, max_splits() / a.nwin);
    set_splits(a, ssp);
    splits = a.nwin * a.slow_splits;
    TENRSO_TRY(partial_buffer(splits, &partial));
    if (with_norm) {
      void* np = nullptr;
      nnorm = (int)(rtiles * splits * waves);
      TENRSO_TRY(ctx_buffer(ctx, SLOT_NORM, (size_t)nnorm * sizeof(double), &np));
      a.norm = (double*)np;
      norm = a.norm;
    }
    if (job && !fuse_job) TENRSO_TRY(als_job_launch(ctx, *job));
    const dim3 block(waves * 64);
    // BF16 with the job fused: the MTTKRP workgroups wait for the job's Gram loads
    // (the job, not the MTTKRP, sets the length of that launch; an fp32 launch only
    // gets longer: 19.2 us without the gate, 22.1 with it, at 256^3 rank 64)
    unsigned* gate = nullptr;
    if (!fp32 && fuse_job && ctx->job_gate) {
      void* gp = nullptr;
      TENRSO_TRY(ctx_buffer(ctx, SLOT_GATE, sizeof(unsigned), &gp));
      gate = (unsigned*)gp;
    }
    auto launch_main = [&](bool with_job) -> int {
      for (int rc = 0; rc < rchunks; ++rc) {
        const int has_job = (with_job && fuse_job && rc == 0) ? 1 : 0;
        AlsJob jarg{};
        if (has_job) {
          jarg = *job;
          if (gate) {
            jarg.gate = gate;
            jarg.gate_stamp = ++ctx->gate_stamp;
          }
        }
        a.r0 = rc * RT;
        a.rcount = (int)std::min<i64>(RT, R - a.r0);
        // (a matrix of tens of millions of rows has more tiles than a launch takes)
        for (i64 t0 = 0; t0 < rtiles * splits; t0 += MAX_THREADS / block.x - 1) {
          int hj = t0 == 0 ? has_job : 0;
          const i64 tiles_now = std::min<i64>(rtiles * splits - t0, MAX_THREADS / block.x - 1);
          a.tile0 = (int)t0;
          void* args[] = {(void*)&Xuse, &a, &partial, &jarg, &hj};
          TENRSO_HIP_TRY(hipLaunchKernel(kern, dim3((unsigned)(tiles_now + hj)), block, args, 0, ctx->stream));
        }
      }
      return TENRSO_OK;
    };
    if (ctx->profile_reps > 0) {
      // profiling: the main kernel alone, `profile_reps` times between two events
      TENRSO_TRY(launch_main(true));
      TENRSO_HIP_TRY(hipEventRecord(ctx->ev0, ctx->stream));
      for (int rep = 0; rep < ctx->profile_reps; ++rep) TENRSO_TRY(launch_main(false));
      TENRSO_HIP_TRY(hipEventRecord(ctx->ev1, ctx->stream));
      TENRSO_HIP_TRY(hipEventSynchronize(ctx->ev1));
      float ms = 0.f;
      TENRSO_HIP_TRY(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
      ctx->last_kernel_ms = (double)ms / ctx->profile_reps;
    } else {
      TENRSO_TRY(launch_main(true));
    }
  } else {
    if (plan) return TENRSO_OK;
    if (pad > 0 && fast_stride != pl.fast_size) {
      set_error("internal: a padded tensor copy reached the generic MTTKRP");
      return TENRSO_ERR_UNSUPPORTED;
    }
    if (job) TENRSO_TRY(als_job_launch(ctx, *job));
    GenericArgs ga{};
    ga.nd = nd;
    ga.mode = mode_use;
    ga.n_oth = pl.n_oth;
    ga.I = I;
    ga.Q = pl.Q;
    ga.R = R;
    ga.J = pl.J;
    for (int m = 0; m < pl.n_oth; ++m) {
      ga.oth_size[m] = pl.oth_size[m];
      ga.oth_fac[m] = Fv[pl.oth[m]];
    }
    ga.bf16 = (bf16 && !x3) ? 1 : 0;
    const i64 tiles = cdiv(nout, 256);
    splits = (int)std::max<i64>(1, std::min<i64>(pl.J, (2LL * ctx->num_cus + tiles - 1) / std::max<i64>(1, tiles)));
    splits = std::min(splits, 1024);
    if (max_splits() < 1) return too_small(1);
    splits = (int)std::min<i64>(splits, max_splits());
    ga.splits = splits;
    TENRSO_TRY(partial_buffer(splits, &partial));
    if (nout > 0) {
      hipLaunchKernelGGL(mttkrp_generic, dim3((unsigned)tiles, splits), dim3(256), 0, ctx->stream, Xuse, ga,
                         partial);
      TENRSO_HIP_TRY(hipGetLastError());
    }
  }

  if (res) {
    res->partial = partial;
    res->splits = splits;
    res->norm = norm;
    res->nnorm = nnorm;
  }
  if (outk == MttkrpOut::F32) return reduce_partials(ctx, partial, splits, nout, (float*)out, nullptr);
  if (outk == MttkrpOut::F64) return reduce_partials(ctx, partial, splits, nout, nullptr, (double*)out);
  return TENRSO_OK;
}

// All modes in one launch of the fp32 MFMA kernel and one reduction (from four modes on
// one launch for the Khatri-Rao rows before); where a mode cannot run so (rank above
// 64, a last mode of one row), a launch a mode and one reduction.  Small tensors are
// bound by the host and the gaps between launches.  All modes of 64^3 rank 8: 49 us as
// three calls of two launches, 22 with a launch a mode, 15 so; 256^3 rank 64: 61.5,
// 58.4 and 44 us (250^3: 73.5, 70.7, 51; 96^4 rank 32: 260, 248, 202).
int mttkrp_all_modes(tenrso_ctx* ctx, const float* X, int nd, const i64* shape, const float* const* F, i64 R,
                     float* const* outs) {
  static_assert(SLOT_PARTIAL_MODE_END - SLOT_PARTIAL_MODE + 1 == MAXD, "a buffer of partials per mode");
  int modes[MAXD];
  const float* pre[MAXD] = {};
  i64 total = 1, rows = 0;  // elements of X; Khatri-Rao elements of all modes
  for (int m = 0; m < nd; ++m) total *= shape[m];
  for (int m = 0; m < nd; ++m) {
    modes[m] = m;
    rows += total / (shape[m] * shape[m == nd - 1 ? nd - 2 : nd - 1]) * R;
  }
  // (rows far larger than X, as many small modes have, are formed a mode at a time)
  const bool batch = nd >= 4 && rows <= 2 * total;
  if (batch) TENRSO_TRY(mttkrp_pre_batch(ctx, nd, shape, F, R, nd, modes, false, pre));
  ReduceMany r{};
  auto add = [&](int m, const float* partial, int splits) {
    r.part[m] = partial;
    r.splits[m] = splits;
    r.n[m] = shape[m] * R;
    r.out[m] = outs[m];
    r.first[m + 1] = r.first[m] + cdiv(shape[m] * R, 64);
    r.count = m + 1;
  };
  X3Plan plan[MAXD];
  bool one = nd < 4 || batch, wv = true;
  for (int m = 0; one && m < nd; ++m) {
    one = nd < 4 || pre[m] != nullptr;
    if (!one) break;
    TENRSO_TRY(mttkrp_dense(ctx, TENRSO_PREC_FP32, X, nullptr, nd, shape, F, R, m, MttkrpOut::PARTIAL, nullptr, nullptr,
                            nullptr, nullptr, 0, 0, pre[m], false, SLOT_PARTIAL, &plan[m]));
    one = plan[m].ok && plan[m].case_b == (m == nd - 1) && plan[m].xl == plan[m < nd - 1 ? 0 : m].xl;
    wv = wv && plan[m].a.win_vec;
  }
  i64 tiles = 64 * ctx->num_cus;  // a bound of the workgroups of one launch
  for (int m = 0; one && m < nd; ++m) tiles += (i64)plan[m].a.rtiles * plan[m].a.nwin;
  if (one && tiles < MAX_THREADS / 256) {
    const void* kern = mttkrp_x3_kernel_all(plan[0].nt, wv, plan[0].xl, plan[nd - 1].xl);
    int occ = 0;
    TENRSO_TRY(occupancy(ctx, kern, 256, &occ));
    // Splits: the resident workgroups of one round shared between the modes, at least a
    // block a wave (256^3 rank 64: 43.9 us in one round, 48.7 in two, 54.6 in three,
    // 61.4 in one with a few workgroups over).
    // Resident workgroups a CU: three of the registers' four (96^4 rank 32: 200 us against
    // 206 with four and 201 with two), two where X is read at any alignment (250^3 rank 16
    // 42 against 46 with three, 80x90x100x110 rank 30 263 against 304).
    const int most = plan[0].xl == 0 ? 3 : 2;
    const i64 target = (i64)(ctx->wg_per_cu_f32 > 0 ? ctx->wg_per_cu_f32 : std::min(occ, most)) * ctx->num_cus;
    AllModesArgs p{};
    p.nd = nd;
    for (int m = 0; m < nd; ++m) {
      KernArgs& a = plan[m].a;
      const i64 wgs1 = (i64)a.rtiles * a.nwin, nkb = (a.kw + 31) / 32;
      i64 ssp = std::min<i64>(target / (nd * wgs1), a.n_slow * nkb / 4);
      ssp = std::max<i64>(1, std::min<i64>(std::min<i64>(ssp, a.n_slow), 65535 / a.nwin));
      set_splits(a, ssp);
      const int splits = a.nwin * a.slow_splits;
      void* pp = nullptr;
      TENRSO_TRY(ctx_buffer(ctx, SLOT_PARTIAL_MODE + m, (size_t)splits * shape[m] * R * sizeof(float), &pp));
      p.a[m] = a;
      p.partial[m] = (float*)pp;
      p.first[m + 1] = p.first[m] + (unsigned)(a.rtiles * splits);
      add(m, p.partial[m], splits);
    }
    void* args[] = {(void*)&X, &p};
    TENRSO_HIP_TRY(hipLaunchKernel(kern, dim3(p.first[nd]), dim3(256), args, 0, ctx->stream));
  } else {
    for (int m = 0; m < nd; ++m) {
      MttkrpResult res;
      TENRSO_TRY(mttkrp_dense(ctx, TENRSO_PREC_FP32, X, nullptr, nd, shape, F, R, m, MttkrpOut::PARTIAL, nullptr, &res,
                              nullptr, nullptr, 0, 0, pre[m], false, SLOT_PARTIAL_MODE + m));
      add(m, res.partial, res.splits);
    }
  }
  hipLaunchKernelGGL(reduce_many_kernel, dim3(r.first[r.count]), dim3(64 * RED_GROUPS), 0, ctx->stream, r);
  TENRSO_HIP_TRY(hipGetLastError());
  return TENRSO_OK;
}

}  // namespace tenrso
