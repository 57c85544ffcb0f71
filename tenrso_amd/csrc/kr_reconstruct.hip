// kr_reconstruct.hip -- Khatri-Rao product and CP reconstruction kernels.
//
// khatri_rao  (tenrso-kernels/src/khatri_rao.rs:56-89): C[ia*J + ib, k] = A[ia,k] * B[ib,k]
//   One rounding per element, so the result is bit-identical to the reference's
//   serial / parallel / blocked variants.  Write-bound: each thread produces 4
//   consecutive k of one output row (16-byte stores when K % 4 == 0).
// cp_reconstruct (tenrso-kernels/src/outer.rs:223-274):
//   out[i_0..i_{N-1}] = sum_r (prod_k F_k[i_k, r]) * w_r.
//   An FP32 matrix product of two Khatri-Rao factors formed in LDS.
#include <algorithm>
#include <cfloat>
#include <type_traits>

#include "kr_reconstruct.hpp"

namespace tenrso {

typedef float floatx4 __attribute__((ext_vector_type(4)));

static inline unsigned cdiv(i64 a, i64 b) { return (unsigned)((a + b - 1) / b); }

// vec: K % 4 == 0 and A, B, C 16-byte aligned (checked on the host): 16-byte
// loads and stores, else scalar
__global__ __launch_bounds__(256) void khatri_rao_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                         i64 I, i64 J, i64 K, float* __restrict__ C, int vec) {
  const i64 t = (i64)blockIdx.x * 256 + threadIdx.x;
  const i64 kq = (K + 3) / 4;
  if (t >= I * J * kq) return;
  const i64 row = t / kq, k0 = (t - row * kq) * 4;
  const i64 ia = row / J, ib = row - ia * J;
  const float* a = A + ia * K;
  const float* b = B + ib * K;
  float* c = C + row * K;
  if (vec && k0 + 3 < K) {
    const float4 av = *reinterpret_cast<const float4*>(a + k0);
    const float4 bv = *reinterpret_cast<const float4*>(b + k0);
    *reinterpret_cast<float4*>(c + k0) = make_float4(av.x * bv.x, av.y * bv.y, av.z * bv.z, av.w * bv.w);
  } else {
    for (i64 k = k0; k < K && k < k0 + 4; ++k) c[k] = a[k] * b[k];
  }
}

int khatri_rao_f32(tenrso_ctx* ctx, const float* A, i64 I, const float* B, i64 J, i64 K, float* C) {
  const i64 n = I * J * ((K + 3) / 4);
  if (n == 0) return TENRSO_OK;
  const int vec = K % 4 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)B % 16 == 0 && (uintptr_t)C % 16 == 0;
  hipLaunchKernelGGL(khatri_rao_kernel, dim3(cdiv(n, 256)), dim3(256), 0, ctx->stream, A, B, I, J, K, C, vec);
  TENRSO_HIP_TRY(hipGetLastError());
  return TENRSO_OK;
}

struct ReconArgs {
  int nd, h;           // modes [0, h) are the rows of the output matrix, [h, nd) its columns
  i64 R, M, N;         // M = product of the row modes, N of the column modes
  i64 shape[MAXD_RECON];
  const float* F[MAXD_RECON];
  const float* w;
  int vec;              // R % 4 == 0 and every factor 16-byte aligned: 16-byte factor loads
  unsigned ctiles;
  unsigned tile0;       // the launch's first tile
  const float* xsub;    // not null: out = xsub - reconstruction (a residual)
  const float* gscale;  // not null: out *= gscale[0] (a device scalar)
};

// out (M x N) = KR(F_0..F_{h-1}) diag(w) KR(F_h..F_{nd-1})^T as an FP32 matrix-core
// product (v_mfma_f32_16x16x4f32).  A workgroup of 4 waves owns a TILE x TILE
// tile (TILE = 32 T, a wave 16T x 16T of it): it forms the Khatri-Rao rows of its
// rows and of its columns in LDS, KT ranks at a time (products left to right, one
// rounding each), and contracts them.  Ranks past R are zero on both sides.  The
// columns are the M dimension of the instruction, so a lane ends with four
// consecutive output elements and stores 16 bytes (VS: N % 4 == 0 and aligned).
// Operands are read from LDS as 4 consecutive ranks (lane group g, step s
// contracts rank 16u + 4g + s on both sides); the pitch of KT + 4 floats keeps
// those 16-byte reads free of bank conflicts.
// A product of one side alone may leave the exponent range where the whole product,
// left to right, does not (factors of sizes 1e30, 1e-25, 1e-25).  Every thread keeps
// the extremes of its products; where one is subnormal or not finite although its
// factors are neither zero nor infinite, and the other side could bring it back, the
// tile is formed again element by element.
// Bound: at 256^3 rank 64 the 2.1 GFLOP take 14 us at the matrix cores' FP32
// peak and the 64 MiB of output 13 us at 5.2 TB/s; the form with one thread per
// element, each lane reading factor rows at a stride of R floats, took 2580 us; this
// one takes 28 us (76 TFLOP/s).
template <int KT, int T, bool VS>
__global__ __launch_bounds__(256) void reconstruct_kernel(ReconArgs a, float* __restrict__ out) {
  constexpr int TILE = 32 * T, PITCH = KT + 4;
  __shared__ __attribute__((aligned(16))) float sk[2 * TILE * PITCH];  // rows, then columns
  __shared__ i64 sidx[MAXD_RECON][TILE];
  __shared__ int range;  // 1, 2: a product of the rows, columns is subnormal; 4, 8: one is above 1; 16: not finite
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  const unsigned tile = a.tile0 + blockIdx.x;
  const i64 r_base = (i64)(tile / a.ctiles) * TILE, c_base = (i64)(tile % a.ctiles) * TILE;
  // factor rows of every tile row (modes < h) and column (modes >= h); those past
  // the end repeat the last one and are not stored
  if (tid == 0) range = 0;
  if (tid < 2 * TILE) {
    const bool col = tid >= TILE;
    const int e = col ? tid - TILE : tid;
    i64 rem = col ? (c_base + e < a.N ? c_base + e : a.N - 1) : (r_base + e < a.M ? r_base + e : a.M - 1);
    for (int k = (col ? a.nd : a.h) - 1; k >= (col ? a.h : 0); --k) {
      sidx[k][e] = rem % a.shape[k];
      rem /= a.shape[k];
    }
  }
  floatx4 acc[T][T];  // [column tile][row tile]
#pragma unroll
  for (int j = 0; j < T; ++j)
#pragma unroll
    for (int i = 0; i < T; ++i) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
  const float* sr = sk + (16 * T * (wave >> 1) + c) * PITCH + 4 * g;
  const float* sc = sk + (TILE + 16 * T * (wave & 1) + c) * PITCH + 4 * g;
  int seen = 0;  // bits of `range`
  float big[2] = {0.f, 0.f};
  for (i64 r0 = 0; r0 < a.R; r0 += KT) {
    __syncthreads();  // indices written, or the previous chunk read
    // one side at a time: a thread's units (4 ranks of one row each) load their
    // rows of one factor together
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      constexpr int UN = TILE * (KT / 4) / 256;
      const int q4 = 4 * (tid % (KT / 4));
      const i64 r = r0 + q4;
      floatx4 v[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) v[u] = floatx4{1.f, 1.f, 1.f, 1.f};
      const int k0 = side ? a.h : 0, k1 = side ? a.nd : a.h;
      for (int k = k0; k < k1; ++k) {
        const float* Fk = a.F[k];
        if (a.vec) {
          const i64 rr = r < a.R ? r : 0;  // ranks past R are zeroed below
#pragma unroll
          for (int u = 0; u < UN; ++u)
            v[u] *= *reinterpret_cast<const floatx4*>(Fk + sidx[k][(tid + 256 * u) / (KT / 4)] * a.R + rr);
        } else {
#pragma unroll
          for (int u = 0; u < UN; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q)
              v[u][q] *= Fk[sidx[k][(tid + 256 * u) / (KT / 4)] * a.R + (r + q < a.R ? r + q : 0)];
        }
      }
      float wq[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) wq[q] = (a.w && side == 0 && r + q < a.R) ? a.w[r + q] : 1.f;
      float least = 1.f, zeros = 0.f;  // zeros: NaN where a product is not finite
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        floatx4 sv;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          v[u][q] = r + q < a.R ? v[u][q] * wq[q] : 1.f;
          sv[q] = r + q < a.R ? v[u][q] : 0.f;
          least = fminf(least, fabsf(v[u][q]));
          big[side] = fmaxf(big[side], fabsf(v[u][q]));
          zeros = fmaf(v[u][q], 0.f, zeros);
        }
        *reinterpret_cast<floatx4*>(sk + (side * TILE + (tid + 256 * u) / (KT / 4)) * PITCH + q4) = sv;
      }
      if (least < 0x1p-126f || !(zeros == 0.f)) {
#pragma unroll 1
        for (int x = 0; x < UN * 4; ++x) {
          const i64 rx = r + x % 4;
          if (rx >= a.R) continue;
          bool nonzero = true, finite = true;
          float p = 1.f;
          for (int k = k0; k < k1; ++k) {
            const float f = a.F[k][sidx[k][(tid + 256 * (x / 4)) / (KT / 4)] * a.R + rx];
            nonzero = nonzero && f != 0.f;
            finite = finite && fabsf(f) <= FLT_MAX;
            p *= f;
          }
          if (a.w && side == 0) {
            const float f = a.w[rx];
            nonzero = nonzero && f != 0.f;
            finite = finite && fabsf(f) <= FLT_MAX;
            p *= f;
          }
          if (nonzero && fabsf(p) < 0x1p-126f) seen |= 1 << side;
          if (finite && !(fabsf(p) <= FLT_MAX)) seen |= 16;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < KT / 16; ++u) {
      floatx4 rv[T], cv[T];
#pragma unroll
      for (int i = 0; i < T; ++i) {
        rv[i] = *reinterpret_cast<const floatx4*>(sr + 16 * i * PITCH + 16 * u);
        cv[i] = *reinterpret_cast<const floatx4*>(sc + 16 * i * PITCH + 16 * u);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < T; ++j)
#pragma unroll
          for (int i = 0; i < T; ++i)
            acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(cv[j][s], rv[i][s], acc[j][i], 0, 0, 0);
    }
  }
  if (big[0] > 1.f) seen |= 4;
  if (big[1] > 1.f) seen |= 8;
#pragma unroll
  for (int b = 0; b < 5; ++b)
    if (__any(seen >> b & 1) && lane == 0) atomicOr(&range, 1 << b);
  __syncthreads();
  const float gs = a.gscale ? a.gscale[0] : 1.0f;
  if ((range & 16) || ((range & 1) && (range & 8)) || ((range & 2) && (range & 4))) {
    int x0 = tid;
    asm volatile("" : "+v"(x0));  // (nothing of this in registers during the loop above)
#pragma unroll 1
    for (int x = x0; x < TILE * TILE; x += 256) {
      const i64 row = r_base + x / TILE, col = c_base + x % TILE;
      if (row >= a.M || col >= a.N) continue;
      float s = 0.f;
#pragma unroll 1
      for (i64 r = 0; r < a.R; ++r) {
        float p = 1.f;
        for (int k = 0; k < a.nd; ++k) p *= a.F[k][sidx[k][k < a.h ? x / TILE : x % TILE] * a.R + r];
        if (a.w) p *= a.w[r];
        s += p;
      }
      const i64 o = row * a.N + col;
      if (a.xsub) s = a.xsub[o] - s;
      if (a.gscale) s *= gs;
      out[o] = s;
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const i64 row = r_base + 16 * T * (wave >> 1) + 16 * i + c;
    if (row >= a.M) continue;
#pragma unroll
    for (int j = 0; j < T; ++j) {
      const i64 col = c_base + 16 * T * (wave & 1) + 16 * j + 4 * g;
      const i64 o = row * a.N + col;
      floatx4 v = acc[j][i];
      if constexpr (VS) {
        if (col < a.N) {
          if (a.xsub) v = *reinterpret_cast<const floatx4*>(a.xsub + o) - v;
          if (a.gscale) v *= gs;
          *reinterpret_cast<floatx4*>(out + o) = v;
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (col + q < a.N) {
            float x = v[q];
            if (a.xsub) x = a.xsub[o + q] - x;
            if (a.gscale) x *= gs;
            out[o + q] = x;
          }
        }
      }
    }
  }
}

int cp_reconstruct_f32(tenrso_ctx* ctx, int nd, const i64* shape, const float* const* F, i64 R, const float* w,
                       float* out) {
  return cp_residual_f32(ctx, nd, shape, F, R, w, nullptr, nullptr, out);
}

int cp_residual_f32(tenrso_ctx* ctx, int nd, const i64* shape, const float* const* F, i64 R, const float* w,
                    const float* X, const float* gscale, float* out) {
  ReconArgs a{};
  a.xsub = X;
  a.gscale = gscale;
  a.nd = nd;
  a.R = R;
  a.w = w;
  a.vec = R % 4 == 0;
  i64 total = 1;
  for (int k = 0; k < nd; ++k) {
    a.shape[k] = shape[k];
    a.F[k] = F[k];
    a.vec = a.vec && (uintptr_t)F[k] % 16 == 0;
    total *= shape[k];
  }
  if (total == 0) return TENRSO_OK;
  // The split of the modes into rows and columns of the output matrix that needs
  // the fewest tiles (the later of equal ones: more factor rows shared by a
  // workgroup's columns), for 128 x 128 tiles, or 64 x 64 ones where those are
  // fewer than the CUs (64^3 rank 8: 32 tiles of 128 against 64 of 64).
  i64 best = 0;
  int tile = 128;
  for (int pass = 0; pass < 2; ++pass) {
    best = 0;
    i64 M = 1;
    for (int h = 0; h <= nd; ++h) {
      const i64 N = total / M, tiles = ((M + tile - 1) / tile) * ((N + tile - 1) / tile);
      if (best == 0 || tiles <= best) {
        best = tiles;
        a.h = h;
        a.M = M;
        a.N = N;
      }
      if (h < nd) M *= shape[h];
    }
    if (pass == 1 || best >= ctx->num_cus) break;
    tile = 64;
  }
  if (best > (i64)INT32_MAX) {
    set_error("reconstruction of %lld elements exceeds the launch bound", (long long)total);
    return TENRSO_ERR_UNSUPPORTED;
  }
  a.ctiles = cdiv(a.N, tile);
  const bool vs = a.N % 4 == 0 && (uintptr_t)out % 16 == 0 && (!X || (uintptr_t)X % 16 == 0);
  auto launch = [&](auto kt, auto t) {
    // (a vector of 2^31 elements has more tiles than the 2^32 - 1 threads of a launch)
    constexpr i64 MOST = UINT32_MAX / 256;
    for (i64 t0 = 0; t0 < best; t0 += MOST) {
      a.tile0 = (unsigned)t0;
      const dim3 grid((unsigned)std::min<i64>(MOST, best - t0));
      if (vs)
        hipLaunchKernelGGL((reconstruct_kernel<decltype(kt)::value, decltype(t)::value, true>), grid, dim3(256), 0,
                           ctx->stream, a, out);
      else
        hipLaunchKernelGGL((reconstruct_kernel<decltype(kt)::value, decltype(t)::value, false>), grid, dim3(256), 0,
                           ctx->stream, a, out);
    }
  };
  auto by_rank = [&](auto t) {
    if (R <= 16) launch(std::integral_constant<int, 16>{}, t);
    else if (R <= 32) launch(std::integral_constant<int, 32>{}, t);
    else launch(std::integral_constant<int, 64>{}, t);
  };
  if (tile == 128) by_rank(std::integral_constant<int, 4>{});
  else by_rank(std::integral_constant<int, 2>{});
  TENRSO_HIP_TRY(hipGetLastError());
  return TENRSO_OK;
}

// ---- extract_weights (cp/types.rs:421-446) ----------------------------------
// For every factor k and column r: n = ||F_k[:, r]||; where n > f32 epsilon the
// column is divided by n and w_r is multiplied by n (w starts at ones).  The
// norms are formed in FP64 (squares of the fp32 entries, fixed order), rounded to
// fp32 for the division, as the reference's f32 instantiation divides by its f32
// norm.  One workgroup per (factor, 64-column block): 16 row lanes x 64 columns,
// each row lane sums rows lane, lane + 16, ...; the 16 sums are added in lane
// order in LDS.  A second launch multiplies the weights in factor order.
struct NormArgs {
  float* F[MAXD_RECON];
  i64 rows[MAXD_RECON];
};

constexpr int EW_COLS = 64, EW_LANES = 16;

__global__ __launch_bounds__(EW_COLS* EW_LANES) void column_normalize_kernel(NormArgs a, i64 R, int cblocks,
                                                                              double* __restrict__ norms) {
  __shared__ double part[EW_LANES][EW_COLS];
  __shared__ float scale[EW_COLS];
  const int k = blockIdx.x / cblocks;
  const i64 c = (i64)(blockIdx.x - k * cblocks) * EW_COLS + (threadIdx.x % EW_COLS);
  const int lane = threadIdx.x / EW_COLS;
  float* __restrict__ F = a.F[k];
  const i64 I = a.rows[k];
  double s = 0.0;
  if (c < R)
    for (i64 i = lane; i < I; i += EW_LANES) {
      const double v = F[i * R + c];
      s += v * v;
    }
  part[lane][threadIdx.x % EW_COLS] = s;
  __syncthreads();
  if (lane == 0) {
    double t = 0.0;
    for (int l = 0; l < EW_LANES; ++l) t += part[l][threadIdx.x];
    const double n = sqrt(t);
    const bool keep = n > (double)__FLT_EPSILON__;
    scale[threadIdx.x] = keep ? (float)n : 0.0f;
    if (c < R) norms[(i64)k * R + c] = keep ? n : 1.0;
  }
  __syncthreads();
  const float n = scale[threadIdx.x % EW_COLS];
  if (c < R && n != 0.0f)
    for (i64 i = lane; i < I; i += EW_LANES) F[i * R + c] = F[i * R + c] / n;
}

__global__ __launch_bounds__(256) void weights_from_norms_kernel(const double* __restrict__ norms, int nd, i64 R,
                                                                 float* __restrict__ w) {
  const i64 r = (i64)blockIdx.x * 256 + threadIdx.x;
  if (r >= R) return;
  double p = 1.0;
  for (int k = 0; k < nd; ++k) p *= norms[(i64)k * R + r];
  w[r] = (float)p;
}

int cp_extract_weights_f32(tenrso_ctx* ctx, int nd, const i64* shape, float* const* F, i64 R, float* w) {
  if (R == 0) return TENRSO_OK;
  NormArgs a{};
  for (int k = 0; k < nd; ++k) {
    a.F[k] = F[k];
    a.rows[k] = shape[k];
  }
  void* norms;
  TENRSO_TRY(ctx_buffer(ctx, SLOT_TMP2, (size_t)nd * R * sizeof(double), &norms));
  const int cblocks = (int)cdiv(R, EW_COLS);
  hipLaunchKernelGGL(column_normalize_kernel, dim3(nd * cblocks), dim3(EW_COLS * EW_LANES), 0, ctx->stream, a, R,
                     cblocks, (double*)norms);
  TENRSO_HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(weights_from_norms_kernel, dim3(cdiv(R, 256)), dim3(256), 0, ctx->stream,
                     (const double*)norms, nd, R, w);
  TENRSO_HIP_TRY(hipGetLastError());
  return TENRSO_OK;
}

}  // namespace tenrso
