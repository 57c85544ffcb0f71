// mttkrp_tile.hpp -- what the MFMA MTTKRP kernels share: their arguments, the LDS
// window of the fastest mode, the block schedule of a wave and the fixed-order
// reduction of a workgroup.
#pragma once
#include <type_traits>

#include "als_job.hpp"
#include "mttkrp.hpp"

namespace tenrso {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx8 __attribute__((ext_vector_type(8)));
typedef uint32_t uint32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t uint32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

struct KernArgs {
  i64 I, Q;           // X viewed as [P, I, Q]
  i64 R;              // factor row stride (rank)
  i64 fast_size;      // size of the fastest other mode
  i64 fast_stride;    // its extent in memory: fast_size, or more in a copy whose last
                      // mode is padded (Q is then the padded extent too)
  i64 qs;             // Q / fast_stride: slow indices per p (case A)
  const float* pre;   // PRE (rows = J / fast_size, stride R) or null (= 1)
  const float* fast;  // FAST factor (fast_size x R)
  int kw;             // window of the fastest mode held in LDS (a multiple of the block)
  int nwin;           // windows, ceil(fast_size / kw)
  i64 n_slow;         // J / fast_size
  i64 total;          // elements of X in memory
  int slow_splits;    // splits of the slow range; nwin * slow_splits partials
  i64 slow_q, slow_rem;  // n_slow = slow_q * slow_splits + slow_rem
  int r0;             // first rank column of this launch
  int rcount;         // rank columns handled by the launch (<= 16*NT)
  int rtiles;         // row tiles; workgroup tile -> (tile % rtiles, split = tile / rtiles)
  int tile0;          // the launch's first tile
  double* norm;       // sums of squares of X, one per wave of the launch (NORM kernels)
  int win_vec;        // FAST 16-byte aligned and R % 4 == 0: 16-byte window loads
};

// The MTTKRPs of all modes of a tensor in one launch: mode m takes the workgroups
// [first[m], first[m + 1]); the last mode is case B.
struct AllModesArgs {
  int nd;
  unsigned first[MAXD + 1];
  float* partial[MAXD];
  KernArgs a[MAXD];
};

__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);  // quiet NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// Stage FAST[w*kw .. w*kw+kw) (columns r0 .. r0+RT) into LDS transposed: s[r][kk].
// Work unit u of the workgroup covers ranks r4 .. r4+3 (r4 = 4*(u % (RT/4))) of
// window rows kk = 2*(u / (RT/4)) and kk + 1, so it leaves LDS as one 8-byte
// (fp32) or two 4-byte (bf16 hi, lo) pairs per rank.  With a 16-byte aligned
// FAST and R % 4 == 0 (win_vec) a unit is two 16-byte loads, else eight 4-byte
// loads (one kernel instance per case, so that every instance has a single
// load sequence and the waits stay exact).  Ranks past rcount and rows past kv load
// the first columns of window row 0 instead (always inside FAST), so no load waits for
// a select: those rank columns are never stored, those rows are never read or
// (window_zero_tail) zeroed, and window_min, which does see them, sees values of the
// window.
// Split in two so the window loads are issued before the first X blocks: the
// LDS writes then wait for the window only (vector loads retire in issue order).
template <int RT, int NTH, int KWMAX>
struct FastWindow {
  static constexpr int UNITS = RT / 4 * (KWMAX / 2);
  static constexpr int PERU = (UNITS + NTH - 1) / NTH;
  // every unit index below PERU*NTH maps in bounds: u >= UNITS gives kk >= KWMAX
  static __device__ __forceinline__ bool live(int u) { return UNITS % NTH == 0 || u < UNITS; }
  floatx4 v[PERU][2];
};

// kv: rows of the window that exist (kw, or fewer in the last window of a
// fastest mode that kw does not divide); a row past kv is read as row 0 (always
// inside FAST) and stored as zero by stage_window_store*.
template <bool WV, int RT, int NTH, int KWMAX>
__device__ __forceinline__ void stage_window_load(FastWindow<RT, NTH, KWMAX>& fw, const KernArgs& a, int w, int kv) {
  const float* base = a.fast + (i64)w * a.kw * a.R + a.r0;
  if constexpr (WV) {
#pragma unroll
    for (int e = 0; e < FastWindow<RT, NTH, KWMAX>::PERU; ++e) {
      const int u = threadIdx.x + e * NTH;
      const int r4 = 4 * (u % (RT / 4)), kk = 2 * (u / (RT / 4));
      const bool ok = kk < kv && r4 < a.rcount;
      const bool ok1 = ok && kk + 1 < kv;
      const float* p = base + (ok ? kk * a.R + r4 : 0);
      fw.v[e][0] = *reinterpret_cast<const floatx4*>(p);
      fw.v[e][1] = *reinterpret_cast<const floatx4*>(p + (ok1 ? a.R : 0));
    }
  } else {
#pragma unroll
    for (int e = 0; e < FastWindow<RT, NTH, KWMAX>::PERU; ++e) {
      const int u = threadIdx.x + e * NTH;
      const int r4 = 4 * (u % (RT / 4)), kk = 2 * (u / (RT / 4));
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const bool ok = kk < kv && r4 + q < a.rcount;
        const bool ok1 = ok && kk + 1 < kv;
        const float* p = base + (ok ? kk * a.R + r4 + q : 0);
        fw.v[e][0][q] = p[0];
        fw.v[e][1][q] = p[ok1 ? a.R : 0];
      }
    }
  }
}

// rows kk >= kv of a staged pair are zero (they meet masked, zero X elements)
template <int RT, int NTH, int KWMAX>
__device__ __forceinline__ void window_zero_tail(FastWindow<RT, NTH, KWMAX>& fw, int kv) {
#pragma unroll
  for (int e = 0; e < FastWindow<RT, NTH, KWMAX>::PERU; ++e) {
    const int u = threadIdx.x + e * NTH;
    const int kk = 2 * (u / (RT / 4));
    if (kk >= kv) fw.v[e][0] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (kk + 1 >= kv) fw.v[e][1] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
}

// Smallest over the wave: within rows of 16 lanes, then across them, by DPP (shuffles
// through LDS are six round trips; with two such reductions a launch of 32^3 took 5.9 us
// instead of 5.5).
__device__ __forceinline__ uint32_t wave_min(uint32_t v) {
#define TENRSO_DPP_MIN(CTRL, ROWS) v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, ROWS, 0xf, false))
  TENRSO_DPP_MIN(0x111, 0xf);  // row_shr:1, 2, 4, 8
  TENRSO_DPP_MIN(0x112, 0xf);
  TENRSO_DPP_MIN(0x114, 0xf);
  TENRSO_DPP_MIN(0x118, 0xf);
  TENRSO_DPP_MIN(0x142, 0xa);  // row_bcast:15 into rows 1 and 3, row_bcast:31 into 2 and 3
  TENRSO_DPP_MIN(0x143, 0xc);
#undef TENRSO_DPP_MIN
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The smallest magnitude of the bf16 values that are not zero, kept for each half of a
// word as 2 |v| - 1 in 16 unsigned bits (zero becomes the largest): two instructions a
// pair.
struct MinNonzero {
  typedef unsigned short ushortx2 __attribute__((ext_vector_type(2)));
  ushortx2 m = {0xffff, 0xffff};
  __device__ __forceinline__ void add(uint32_t pair) {
    uint32_t two = 0x00020002u, ones = 0xffffffffu;
    asm("" : "+s"(two), "+s"(ones));  // a multiply-add, not a shift and an add
    const ushortx2 t =
        __builtin_bit_cast(ushortx2, pair) * __builtin_bit_cast(ushortx2, two) + __builtin_bit_cast(ushortx2, ones);
    m = __builtin_elementwise_min(m, t);
  }
  // 2^126 if there is none
  __device__ __forceinline__ float value() const {
    const uint32_t b = ((uint32_t)min(m[0], m[1]) + 1) >> 1;
    return b == 0x8000u ? 0x1p126f : __uint_as_float(b << 16);
  }
};

// The smallest magnitude of the values a wave stages that are not zero, 2^126 if there
// is none.  (Fillers of rows and ranks that do not exist repeat values of the window.)
// Kept as 2 |v| - 1 in unsigned words, which zero makes the largest.
template <int RT, int NTH, int KWMAX>
__device__ __forceinline__ float window_min(const FastWindow<RT, NTH, KWMAX>& fw) {
  uint32_t m = 0xffffffffu;
#pragma unroll
  for (int e = 0; e < FastWindow<RT, NTH, KWMAX>::PERU; ++e)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < 4; ++q) m = min(m, (__float_as_uint(fw.v[e][h][q]) << 1) - 1);
  m = wave_min(m);
  return m == 0xffffffffu ? 0x1p126f : __uint_as_float((m >> 1) + 1);
}

// The window in LDS as a bf16 pair: FAST = hi + lo with hi = bf16(FAST) and
// lo = bf16(FAST - hi), so hi + lo carries 16 significant bits.
template <int RT, int PITCH, int NTH, int KWMAX>
__device__ __forceinline__ void stage_window_store_bf16x2(uint16_t* __restrict__ shi, uint16_t* __restrict__ slo,
                                                          const FastWindow<RT, NTH, KWMAX>& fw) {
  static_assert(PITCH % 2 == 0, "pairs of window rows are stored as 4-byte words");
#pragma unroll
  for (int e = 0; e < FastWindow<RT, NTH, KWMAX>::PERU; ++e) {
    const int u = threadIdx.x + e * NTH;
    const int r4 = 4 * (u % (RT / 4)), kk = 2 * (u / (RT / 4));
    if (!FastWindow<RT, NTH, KWMAX>::live(u)) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // v_cvt_pk_bf16_f32 rounds to nearest even, as f32_to_bf16_rne does for
      // every non-NaN value; element 0 (row kk) is the low half
      const floatx2 f = {fw.v[e][0][q], fw.v[e][1][q]};
      const uint32_t hw = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
      const floatx2 r = {f[0] - __uint_as_float(hw << 16), f[1] - __uint_as_float(hw & 0xffff0000u)};
      const uint32_t lw = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
      const int o = (r4 + q) * PITCH + kk;
      *reinterpret_cast<uint32_t*>(&shi[o]) = hw;
      *reinterpret_cast<uint32_t*>(&slo[o]) = lw;
    }
  }
}

// The same as an exact bf16 triple: FAST = hi + lo + lo2 (hi = bf16(FAST),
// lo = bf16(FAST - hi), lo2 = bf16(FAST - hi - lo)); each residual is exact in
// fp32 and the last one has at most 8 significant bits, so for every normal
// fp32 value hi + lo + lo2 equals FAST exactly.
template <int RT, int PITCH, int NTH, int KWMAX>
__device__ __forceinline__ void stage_window_store_bf16x3(uint16_t* __restrict__ shi, uint16_t* __restrict__ slo,
                                                          uint16_t* __restrict__ slo2,
                                                          const FastWindow<RT, NTH, KWMAX>& fw) {
  static_assert(PITCH % 2 == 0, "pairs of window rows are stored as 4-byte words");
#pragma unroll
  for (int e = 0; e < FastWindow<RT, NTH, KWMAX>::PERU; ++e) {
    const int u = threadIdx.x + e * NTH;
    const int r4 = 4 * (u % (RT / 4)), kk = 2 * (u / (RT / 4));
    if (!FastWindow<RT, NTH, KWMAX>::live(u)) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const floatx2 f = {fw.v[e][0][q], fw.v[e][1][q]};
      const uint32_t hw = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
      const floatx2 r = {f[0] - __uint_as_float(hw << 16), f[1] - __uint_as_float(hw & 0xffff0000u)};
      const uint32_t lw = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
      const floatx2 r2 = {r[0] - __uint_as_float(lw << 16), r[1] - __uint_as_float(lw & 0xffff0000u)};
      const uint32_t l2w = __builtin_bit_cast(uint32_t, __builtin_convertvector(r2, bf16x2));
      const int o = (r4 + q) * PITCH + kk;
      *reinterpret_cast<uint32_t*>(&shi[o]) = hw;
      *reinterpret_cast<uint32_t*>(&slo[o]) = lw;
      *reinterpret_cast<uint32_t*>(&slo2[o]) = l2w;
    }
  }
}

// A value the compiler cannot prove uniform but that is: move it to scalar registers.
__device__ __forceinline__ i64 uniform_i64(i64 v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)(uint64_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
  return (i64)(((uint64_t)hi << 32) | lo);
}

// Block loads take their offsets through these, so that each is one unconditional vector
// load.  The compiler otherwise reads a loaded value again from its register where the
// offset may not have changed (after a wait for all loads), and with scalar loads, behind
// a branch, where a wave has no block left: a workgroup's first loads went out one round
// trip after another.
template <bool ON = true>
__device__ __forceinline__ i64 opaque_uniform(i64 v) {
  if constexpr (ON) {
    v = uniform_i64(v);
    asm volatile("" : "+s"(v));
  }
  return v;
}
template <bool ON = true>
__device__ __forceinline__ i64 opaque_lane(i64 v) {
  if constexpr (ON) asm volatile("" : "+v"(v));
  return v;
}

// PRE row used when the MTTKRP has no PRE factor (a matrix): KR = FAST.
#define TENRSO_ONES8 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f
static __device__ float kPreOnes[128] = {
    TENRSO_ONES8, TENRSO_ONES8, TENRSO_ONES8, TENRSO_ONES8, TENRSO_ONES8, TENRSO_ONES8, TENRSO_ONES8, TENRSO_ONES8,
    TENRSO_ONES8, TENRSO_ONES8, TENRSO_ONES8, TENRSO_ONES8, TENRSO_ONES8, TENRSO_ONES8, TENRSO_ONES8, TENRSO_ONES8};
#undef TENRSO_ONES8

// Blocks below b of nkb (1 to 4) a slow index: the slow indices they fill.  Without a
// division by a variable in a workgroup's start (0.15 us of a launch of 24^3).
__device__ __forceinline__ i64 whole_slow(i64 b, int nkb) { return nkb == 3 ? b / 3 : b >> (nkb >> 1); }

// Block schedule of one wave: a contiguous range of the workgroup's blocks, from block
// kb0 of slow index slow0 on, nkb blocks a slow index.  Loads run in that order, so the
// cursor only steps forward, and it stops on the wave's last block (loads past the end
// are redirected by the kernels to one cache line).  Every X and PRE load is thus
// unconditional and the wait before a block's MFMAs counts exactly the loads issued
// after it, which keeps the prefetch in flight.  A wave with no block reads PRE at
// slow index min(slow0, n_slow - 1) and computes nothing.
// Case A (X as [P, I, Q], slow = p*qs + sq): the block starts at element
// p*I*Q + sq*fast_size + w*kw + kb*KB.  Case B: the block covers j = slow*fast_size
// + w*kw + kb*KB onwards, one row of I elements per j.  All fields are uniform.
template <int KB, bool CASE_B>
struct BlockCursor {
  int kb, nkb;
  i64 slow, sq, base, wrap;

  __device__ __forceinline__ BlockCursor(const KernArgs& a, i64 slow0, int w, int nkb_, int kb0) {
    kb = kb0;
    nkb = nkb_;
    slow = slow0 < a.n_slow ? slow0 : a.n_slow - 1;
    if constexpr (!CASE_B) {
      // 32-bit division whenever the slow range fits (it nearly always does)
      const i64 p = (a.n_slow >> 32) ? slow / a.qs : (i64)((uint32_t)slow / (uint32_t)a.qs);
      sq = slow - p * a.qs;
      base = p * a.I * a.Q + sq * a.fast_stride + (i64)w * a.kw;
      wrap = a.I * a.Q - a.qs * a.fast_stride;  // from (p, qs) to (p + 1, 0)
    } else {
      sq = 0;
      wrap = 0;
      base = slow * a.fast_size + (i64)w * a.kw;
    }
  }
  // element offset in X of the block's first element (lane offsets are added on top)
  __device__ __forceinline__ i64 offset(const KernArgs& a) const {
    if constexpr (!CASE_B) return base + (i64)kb * KB;
    else return (base + (i64)kb * KB) * a.I;
  }
  __device__ __forceinline__ void step(const KernArgs& a) {
    if (++kb == nkb) {
      kb = 0;
      ++slow;
      base += a.fast_stride;
      if constexpr (!CASE_B) {
        if (++sq >= a.qs) {
          sq -= a.qs;
          base += wrap;
        }
      }
    }
  }
};

// Fixed-order reduction of the WAVES per-wave accumulators of a workgroup, spread
// over the waves: tile q = mt*NT + nt belongs to wave q % WAVES, which adds the
// WAVES copies of it in wave order 0, 1, .. (one LDS round trip, 16 bytes per
// lane and tile) and stores it; every wave stores its own tiles, so the partial
// leaves the workgroup from all waves at once.  LDS use: MT*NT*WAVES*64 floatx4.
// SYNC: waits first (the LDS window may still be read by other waves).
template <int MT, int NT, int WAVES, bool SYNC = true>
__device__ __forceinline__ void wg_reduce_store(floatx4 (&acc)[MT][NT], float* __restrict__ red, int wave, int lane,
                                                float* __restrict__ out, i64 rows, i64 R, int r0, int rcount,
                                                i64 row_base, bool case_b) {
  floatx4* r4 = reinterpret_cast<floatx4*>(red);
  const int g = lane >> 4, c = lane & 15;
  if constexpr (SYNC) __syncthreads();  // LDS window no longer read
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int q = mt * NT + nt;
      if (q % WAVES != wave) r4[(q * WAVES + wave) * 64 + lane] = acc[mt][nt];
    }
  __syncthreads();
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int q = mt * NT + nt;
      if (q % WAVES != wave) continue;
      floatx4 sum = wave == 0 ? acc[mt][nt] : r4[(q * WAVES + 0) * 64 + lane];
#pragma unroll
      for (int wv = 1; wv < WAVES; ++wv) sum += wv == wave ? acc[mt][nt] : r4[(q * WAVES + wv) * 64 + lane];
      if (16 * nt + c >= rcount) continue;
      const int col = r0 + 16 * nt + c;
      // D layout (16x16): lane (g, c), register v -> tile row 4g + v, column c
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const i64 row = case_b ? row_base + MT * (4 * g + v) + mt : row_base + 16 * mt + 4 * g + v;
        if (row < rows) out[row * R + col] = sum[v];
      }
    }
}

// Fold the per-slow accumulator T into acc with the PRE row of that slow index:
// acc[:, r] += PRE[slow, r] * T[:, r]  (lane (g, c) holds column 16nt + c).
template <int MT, int NT>
__device__ __forceinline__ void fold_slow(floatx4 (&acc)[MT][NT], floatx4 (&T)[MT][NT], const float (&pre)[NT]) {
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      acc[mt][nt] += T[mt][nt] * pre[nt];
      T[mt][nt] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
}

// Zero if every accumulator is finite, else NaN.
template <int MT, int NT>
__device__ __forceinline__ float sum_of_zeros(const floatx4 (&acc)[MT][NT]) {
  float z = 0.f;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int v = 0; v < 4; ++v) z = fmaf(acc[mt][nt][v], 0.f, z);
  return z;
}

// The form of a tile whose values bf16 parts cannot hold: the same blocks again with
// v_mfma_f32_16x16x4_f32, products x (pre fast) in fp32.  The window goes to LDS in
// fp32, s[r][kk] with a pitch of REDO_PITCH; the X blocks are loaded as before, one at a
// time.  A mode of 256^3 at rank 64 takes 24 us, with one NaN in X 45 to 49, with a
// small value in every tile 51 (one thread an output, in turn over the tile's j, took
// 820 to 950 us for the one NaN); the bf16 last mode with infinities in every tile 41
// (1218).
constexpr int REDO_PITCH = 128 + 4;

// (Its addresses are its own: those of stage_window_load would stay in registers
// through the main loop, up to 38 of them.)
template <int RT, int NTH, int KWMAX>
__device__ __forceinline__ void redo_window(float* __restrict__ s, const KernArgs& a, int w, int kv) {
  static_assert(KWMAX + 4 == REDO_PITCH, "rows of the window are 16-byte aligned");
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const float* base = a.fast + (i64)w * a.kw * a.R + a.r0;
#pragma unroll 4
  for (int u = tid; u < RT * KWMAX; u += NTH) {
    const int r = u % RT, kk = u / RT;
    s[r * REDO_PITCH + kk] = kk < kv && r < a.rcount ? base[kk * a.R + r] : 0.f;
  }
}

// acc += x (pre fast) over one block of 32 j: a lane holds eight j of each of its rows,
// from k0 = kb * 32 + 8 g on.
template <int MT, int NT>
__device__ __forceinline__ void redo_block(floatx4 (&acc)[MT][NT], const floatx8 (&x)[MT], const float (&pre)[NT],
                                           const float* __restrict__ s, int c, int k0, int kv) {
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const float* row = s + (16 * nt + c) * REDO_PITCH + k0;
    const floatx4 f0 = *reinterpret_cast<const floatx4*>(row), f1 = *reinterpret_cast<const floatx4*>(row + 4);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      // rows past kv are zero, but pre may be infinite
      const float kr = k0 + e < kv ? pre[nt] * (e < 4 ? f0[e & 3] : f1[e & 3]) : 0.f;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[mt][e], kr, acc[mt][nt], 0, 0, 0);
    }
  }
}

}  // namespace tenrso
