// mttkrp_x3_kernel.hpp -- the fp32 dense MTTKRP on the bf16 matrix cores.
//
// Every fp32 value is an exact sum of three bf16 values (x = x_h + x_l + x_l2), so
// a product x f is six bf16 products down to 2^-16 of the leading one:
//   x_h f_h;  x_h f_l, x_l f_h;  x_h f_l2, x_l f_l, x_l2 f_h
// (what is left out is below 2^-24 of it).  v_mfma_f32_16x16x32_bf16 forms exact
// products and adds them in fp32, sixteen times as fast as the fp32 instruction:
// six terms run at 2.7 times its rate, and the kernel becomes bound by memory.
//
// Measured, one launch, X in memory (256^3 rank 64, 64 MiB): 16.6-18.0 us against
// 26-28 us with v_mfma_f32_16x16x4_f32, whose matrix pipe was busy for 16 us; the
// same launch with one term and no split takes 14.9 us (4.5 TB/s, start and end
// included), the five other terms 2 us more and the split of X 1 us.
//
// Special values.  The split of an infinity, or of a value that rounds to one in
// bf16, gives NaN where fp32 arithmetic gives an infinity or a number.  A value below
// 2^-109 has bits below the last one of any bf16 value (2^-133; denormal operands and
// sums are exact here), and products below 2^-126, which a large PRE may bring back,
// lose bits in T.  Both are seen at the end of the loop (an accumulator that is not
// finite; the smallest magnitudes of X and of the window other than zero, kept on the
// way), and the workgroup then forms its tile again with the fp32 instruction.  The
// smallest, not the largest of a row or column: the large ones may meet zeros.
#pragma once
#include "als_job_wide.hpp"
#include "mttkrp_tile.hpp"

namespace tenrso {

namespace {

// blocks of X in registers: two in flight (three cost registers: 18.6 us against
// 18.0 at 256^3 rank 64), one where eight rank tiles take the registers
template <int NT>
constexpr int X3_NBUF = NT == 8 ? 2 : 3;
constexpr int X3_KWMAX = 128;  // rows of the LDS window

// x - h of a pair, h the pair rounded to bf16: one v_dot2 each (h_0 -1 + h_1 0 + x_0),
// exact, instead of widening h first
__device__ __forceinline__ void x3_residual(const floatx2& x, const bf16x2& h, floatx2& r) {
  uint32_t m0 = 0x0000bf80u, m1 = 0xbf800000u;  // (-1, 0) and (0, -1)
  // in registers: as an inline constant the first would be read as (0, -1)
  asm("" : "+s"(m0), "+s"(m1));
  r[0] = __builtin_amdgcn_fdot2_f32_bf16(h, __builtin_bit_cast(bf16x2, m0), x[0], false);
  r[1] = __builtin_amdgcn_fdot2_f32_bf16(h, __builtin_bit_cast(bf16x2, m1), x[1], false);
}

__device__ __forceinline__ void x3_split(const floatx8& x, bf16x8& h, bf16x8& l, bf16x8& l2) {
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const floatx2 v = {x[2 * p], x[2 * p + 1]};
    floatx2 r, q;
    const bf16x2 hp = __builtin_convertvector(v, bf16x2);
    x3_residual(v, hp, r);
    const bf16x2 lp = __builtin_convertvector(r, bf16x2);
    x3_residual(r, lp, q);
    const bf16x2 l2p = __builtin_convertvector(q, bf16x2);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      h[2 * p + e] = hp[e];
      l[2 * p + e] = lp[e];
      l2[2 * p + e] = l2p[e];
    }
  }
}

// The work split: a workgroup owns 32 rows and one LDS window (up to 128 rows) of the
// fastest mode, its waves contiguous ranges of its blocks (32 consecutive j).  T = X FAST is contracted per slow index and folded
// into the accumulator with PRE[slow].  The FAST window is split once, when it
// goes to LDS; X is split in registers, each element by one wave.
// XL 0: whole windows, 16-byte aligned rows (case B: an even number of rows,
//    8-byte aligned).  XL 4: a zero-padded copy (case A).  XL 1: everything else:
//    16-byte (8-byte in case B) vectors at any 4-byte alignment, which this
//    hardware serves; elements past the window's end are read (they are the next
//    row's) and zeroed, except where that would pass the end of X.
// Forms.  JOB 1: 8 waves and the inlined ALS job, whose registers (235) leave one
// workgroup a CU: the form of launches that carry the job or fill the GPU in one
// round.  JOB 2: the same with the job of ranks 65 to 128, for eight rank tiles (one
// pass over X and one split of it instead of two).  JOB 0: 4 waves: two (NT = 4) to
// four workgroups a CU, so that where a CU runs several one after another the end of one meets the loop of the next
// (9216 rows x 9216 j at rank 32: 69-73 us against 77-85 us; one full round at
// 256^3 rank 64: 19.1 us against 18.4 us).
// NORM: the sum of squares of X as well (FP64; every element of X is read by exactly
// one lane), a partial per wave in a.norm.  In the memory-bound loop it is nearly
// free, where a pass of its own over X takes as long as the MTTKRP.
// ALL: 4 waves, and the workgroups of every mode of the tensor in one launch.

// LDS bytes of the window planes and the reduction
template <int NT, int WAVES>
constexpr int x3_lds() {
  constexpr int win = 3 * 16 * NT * (X3_KWMAX + 8) * 2, red = 2 * NT * WAVES * 64 * 16;
  static_assert(win >= 16 * NT * REDO_PITCH * 4, "the fp32 window of a tile formed again");
  return win > red ? win : red;
}

// One workgroup's tile.  OPAQUE: block loads through opaque_uniform and opaque_lane.
// smem: x3_lds bytes; wmin: smallest magnitude of the window values that each wave
// stages; redo: a wave asks for the fp32 form.
template <int NT, int WAVES, bool CASE_B, bool WV, int XL, bool NORM, bool OPAQUE = true>
__device__ __forceinline__ void x3_tile(const float* __restrict__ X, const KernArgs& a, float* __restrict__ partial,
                                        int tile, float* smem, float* wmin, int& redo) {
  constexpr int MT = 2, NBUF = X3_NBUF<NT>, KWMAX = X3_KWMAX;
  constexpr int KB = 32, PITCH = KWMAX + 8, RT = 16 * NT, NTH = WAVES * 64, ROWS = 16 * MT;
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
  const int kv = XL == 0 ? a.kw : (int)min((i64)a.kw, a.fast_size - (i64)w * a.kw);
  const int nkb = XL == 0 ? a.kw / KB : (kv + KB - 1) / KB;
  // the workgroup's blocks in WAVES contiguous, balanced ranges
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
  double sumsq[MT];  // sum of squares of the lane's rows (NORM)
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) sumsq[mt] = 0.0;
  MinNonzero xmin;  // of the lane's X, rounded to bf16
  struct Buf {
    floatx8 x[MT];
    float pre[NT];
    int kb;
  };

  // per-lane element offsets, fixed for the whole loop; the per-block part of
  // every address is wave-uniform
  // Case A, XL 1: eights of a block that are read.  In a window of one block those past
  // its end are not: their lanes load what the last ones do.
  const int eights = XL == 1 && nkb == 1 ? (kv + 7) / 8 : KB / 8, gl = min(g, eights - 1);
  i64 loff[MT];
  bool tail = false;  // case B, odd I: the lane's row is the second of its pair
  if constexpr (!CASE_B) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const i64 rr = row_base + 16 * mt + c;
      loff[mt] = (rr < a.I ? rr : a.I - 1) * a.Q + 8 * gl;
    }
  } else {
    const i64 rr = row_base + MT * c;
    tail = XL != 0 && rr > a.I - MT;
    loff[0] = (i64)(8 * g) * a.I + (rr <= a.I - MT ? rr : a.I - MT);
  }
  // XL 1: a block starting past `lim` would read past the end of X
  i64 lim = 0;
  if constexpr (XL == 1) {
    const i64 last = (row_base + ROWS < a.I ? row_base + ROWS : a.I) - 1;
    lim = uniform_i64(CASE_B ? a.total - (i64)KB * a.I : a.total - last * a.Q - 8 * eights);
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
    const float* prow = pre_base + opaque_uniform<OPAQUE>(cur.slow * pre_stride);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) b.pre[nt] = prow[poff[nt]];
    // past the last block every lane reads the first elements of X (one cache
    // line): the load stays unconditional and costs the memory pipeline little
    const bool live = t < T;
    const i64 off = opaque_uniform<OPAQUE>(live ? cur.offset(a) : 0);
    const float* ubase = X + off;
    bool inside = true;  // uniform
    if constexpr (XL == 1) inside = live ? off <= lim : a.total >= 8;
    if constexpr (!CASE_B) {
      if (XL != 1 || inside) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const float* base = ubase + opaque_lane<OPAQUE>(live ? loff[mt] : 0);
          floatx4 v0, v1;
          if constexpr (XL == 1) {
            __builtin_memcpy(&v0, __builtin_assume_aligned(base, 4), sizeof(v0));
            __builtin_memcpy(&v1, __builtin_assume_aligned(base + 4, 4), sizeof(v1));
          } else {
            v0 = *reinterpret_cast<const floatx4*>(base);
            v1 = *reinterpret_cast<const floatx4*>(base + 4);
          }
          b.x[mt] = floatx8{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
        }
      } else {
        const int top = live ? kv - 1 - b.kb * KB - 8 * gl : 0;  // past the window's end: its last element
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const float* base = ubase + opaque_lane<OPAQUE>(live ? loff[mt] : 0);
#pragma unroll
          for (int e = 0; e < 8; ++e) b.x[mt][e] = base[min(e, top)];
        }
      }
    } else {
      const float* base = ubase + opaque_lane<OPAQUE>(live ? loff[0] : 0);
      const i64 stride = live ? a.I : 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float* p = base + e * stride;
        if constexpr (XL == 1) {
          if (!inside) p = live && b.kb * KB + 8 * g + e < kv ? p : X;
          float v[2];
          __builtin_memcpy(v, __builtin_assume_aligned(p, 4), sizeof(v));
          b.x[0][e] = v[0];
          b.x[1][e] = v[1];
        } else {
          const float2 v = *reinterpret_cast<const float2*>(p);
          b.x[0][e] = v.x;
          b.x[1][e] = v.y;
        }
      }
    }
    if (t + 1 < T) cur.step(a);
  };

  // eight j of the lane's row mt, zero past the window's end
  auto row_of = [&](const Buf& b, int mt) -> floatx8 {
    floatx8 x = b.x[mt];
    if constexpr (XL == 1) {
      if constexpr (CASE_B) {
        if (mt == 0)
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = tail ? b.x[1][e] : x[e];
      }
      if (b.kb * KB + KB > kv) {  // the window's partly filled last block
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = b.kb * KB + 8 * g + e < kv ? x[e] : 0.f;
      }
    }
    return x;
  };
  auto compute = [&](int t, const Buf& b) {
    if (t >= T) return;
    bf16x8 xh[MT], xl[MT], xl2[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const floatx8 x = row_of(b, mt);
      if constexpr (NORM) {
#pragma unroll
        for (int e = 0; e < 8; ++e) sumsq[mt] = fma((double)x[e], (double)x[e], sumsq[mt]);
      }
      x3_split(x, xh[mt], xl[mt], xl2[mt]);
      const uint32x4 hw = __builtin_bit_cast(uint32x4, xh[mt]);
#pragma unroll
      for (int e = 0; e < 4; ++e) xmin.add(hw[e]);
    }
    // Two rank tiles at a time, term by term (smallest first): consecutive MFMAs
    // then update 2 * MT different accumulators, so none waits for the previous
    // one's result
    constexpr int NG = NT >= 2 ? 2 : 1;
#pragma unroll
    for (int n0 = 0; n0 < NT; n0 += NG) {
      bf16x8 bh[NG], bl[NG], bl2[NG];
#pragma unroll
      for (int u = 0; u < NG; ++u) {
        const int off = (16 * (n0 + u) + c) * PITCH + b.kb * KB + 8 * g;
        bh[u] = *reinterpret_cast<const bf16x8*>(&sHi[off]);
        bl[u] = *reinterpret_cast<const bf16x8*>(&sLo[off]);
        bl2[u] = *reinterpret_cast<const bf16x8*>(&sLo2[off]);
      }
#define TENRSO_X3_TERM(XA, XB)                                                                        \
  _Pragma("unroll") for (int u = 0; u < NG; ++u) _Pragma("unroll") for (int mt = 0; mt < MT; ++mt)     \
      Tacc[mt][n0 + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(XA[mt], XB[u], Tacc[mt][n0 + u], 0, 0, 0);
      TENRSO_X3_TERM(xl2, bh)
      TENRSO_X3_TERM(xl, bl)
      TENRSO_X3_TERM(xh, bl2)
      TENRSO_X3_TERM(xl, bh)
      TENRSO_X3_TERM(xh, bl)
      TENRSO_X3_TERM(xh, bh)
#undef TENRSO_X3_TERM
    }
    // a slow index ends, or this wave's range does (it may end inside one)
    if (b.kb == nkb - 1 || t == T - 1) fold_slow<MT, NT>(acc, Tacc, b.pre);
  };

  Buf b[NBUF];
#pragma unroll
  for (int i = 0; i < NBUF - 1; ++i) load(i, b[i]);
  if constexpr (XL > 0) window_zero_tail(fw, kv);
  const float fw_min = window_min(fw);
  if (lane == 0) wmin[wave] = fw_min;
  stage_window_store_bf16x3<RT, PITCH, NTH, KWMAX>(sHi, sLo, sLo2, fw);
  __syncthreads();  // LDS window staged
  for (int t = 0; t < T; t += NBUF) {
#pragma unroll
    for (int i = 0; i < NBUF; ++i) {
      load(t + i + NBUF - 1, b[(i + NBUF - 1) % NBUF]);
      compute(t + i, b[i]);
    }
  }

  if constexpr (NORM) {
    // rows past I repeat the last one (case B: the last pair)
    double v = 0.0;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const i64 row = CASE_B ? row_base + MT * c + mt : row_base + 16 * mt + c;
      v += row < a.I ? sumsq[mt] : 0.0;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (lane == 0) a.norm[(i64)tile * WAVES + wave] = v;
  }

  // not finite, or too small: all of it again in fp32
  const float xm = xmin.value();  // of the lane
  float fm = wmin[0];
#pragma unroll
  for (int v = 1; v < WAVES; ++v) fm = fminf(fm, wmin[v]);
  const bool small = xm < 0x1p-108f || fm < 0x1p-108f || xm * fm < 0x1p-123f;
  if (__any(small || !(sum_of_zeros<MT, NT>(acc) == 0.f))) redo = 1;
  __syncthreads();
  float* out = partial + (i64)split * a.I * a.R;
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
      const floatx8 x[MT] = {row_of(b[0], 0), row_of(b[0], 1)};
      redo_block(acc, x, b[0].pre, smem, c, b[0].kb * KB + 8 * g, kv);
    }
    __syncthreads();  // window no longer read
  }
  wg_reduce_store<MT, NT, WAVES, false>(acc, smem, wave, lane, out, a.I, a.R, a.r0, a.rcount, row_base, CASE_B);
}

template <int NT, int WAVES, int JOB, bool CASE_B, bool WV, int XL, bool NORM>
__global__ __launch_bounds__(WAVES * 64) void mttkrp_x3_mfma(const float* __restrict__ X, KernArgs a,
                                                             float* __restrict__ partial, AlsJob job, int has_job) {
  constexpr int LDS_B = x3_lds<NT, WAVES>();
  constexpr int LDS_JOB = JOB == 0 ? 0 : (JOB == 1 ? JOB_LDS_BYTES : WIDE_LDS_BYTES);
  constexpr int LDS_BYTES = LDS_B > LDS_JOB ? LDS_B : LDS_JOB;
  __shared__ __attribute__((aligned(16))) float smem[LDS_BYTES / 4];
  __shared__ float wmin[WAVES];
  __shared__ int redo;
  if (JOB != 0 && has_job && blockIdx.x == 0) {
    // one such workgroup a CU, so the job has its CU to itself; waves past the
    // rank-64 job's four end at once
    double* lds = reinterpret_cast<double*>(smem);
    if constexpr (JOB == 1) {
      static_assert((WAVES * 64) % JOB_THREADS == 0, "the ALS job runs on the first 256 threads");
      if (threadIdx.x < JOB_THREADS) als_job_run(job, lds);
    } else if constexpr (JOB == 2) {
      static_assert(WAVES * 64 == WIDE_THREADS, "the wide-rank job runs on the whole workgroup");
      als_job_wide_run(job, lds);
    }
    return;
  }
  x3_tile<NT, WAVES, CASE_B, WV, XL, NORM>(X, a, partial,
                                           a.tile0 + (int)blockIdx.x - (JOB != 0 && has_job ? 1 : 0), smem, wmin, redo);
}

template <int NT, int WAVES, int JOB, bool CASE_B, bool WV, bool NORM>
const void* x3_pick_xl(int xl) {
  if constexpr (!CASE_B && !NORM) {  // (the norm is not taken from a padded copy)
    if (xl == 4) return reinterpret_cast<const void*>(mttkrp_x3_mfma<NT, WAVES, JOB, CASE_B, WV, 4, NORM>);
  }
  if (xl == 0) return reinterpret_cast<const void*>(mttkrp_x3_mfma<NT, WAVES, JOB, CASE_B, WV, 0, NORM>);
  return reinterpret_cast<const void*>(mttkrp_x3_mfma<NT, WAVES, JOB, CASE_B, WV, 1, NORM>);
}

template <int NT, int WAVES, int JOB, bool NORM = false>
const void* x3_pick(bool case_b, bool wv, int xl) {
  if (case_b)
    return wv ? x3_pick_xl<NT, WAVES, JOB, true, true, NORM>(xl) : x3_pick_xl<NT, WAVES, JOB, true, false, NORM>(xl);
  return wv ? x3_pick_xl<NT, WAVES, JOB, false, true, NORM>(xl) : x3_pick_xl<NT, WAVES, JOB, false, false, NORM>(xl);
}

}  // namespace

}  // namespace tenrso
