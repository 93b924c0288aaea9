// qnn_dense.hip -- projections over F32 / BF16 weights (row-major [out, in]).
//
// VectorLinear (Context.Implementation.inc:969-1001; ops GO_LLM_MATVEC /
// GO_LLM_MATVEC_BF16) and Linear with an F32 or BF16 weight
// (Implementation.inc:852-883, the gemm pipeline with the bf16 flag): the
// engine's router projection (LLM.MoE.pas:363-374) and the native-precision
// layers of the models.  bf16 weights widen to fp32 exactly (bits << 16);
// products and sums are fp32.
//
// * one row (dense_matvec_launch): one wave per output row; each lane reads
//   16-byte pieces of the row (4 fp32 or 8 bf16 weights) and the matching
//   activations, two pieces in flight per iteration, then a butterfly sum.
// * fused gate/up SwiGLU, one row (dense_swiglu_launch, op 66): as the
//   matvec, with the gate and up rows of an output read in the same pass.
// * several rows (dense_gemm_launch): fp32 matrix cores (k_dense_mm).
#include "qnn_internal.h"
#include "qnn_lanes.h"

namespace qnn {
namespace {

__device__ __forceinline__ float bf16_to_f32(uint16_t b) { return __uint_as_float(uint32_t(b) << 16); }

// 16-byte piece i of a row as 4 (fp32) or 8 (bf16) floats, dotted with x.
template <bool BF16>
__device__ __forceinline__ float piece_dot(const uint4 w, const float *x) {
  if constexpr (BF16) {
    const uint32_t u[4] = {w.x, w.y, w.z, w.w};
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s = fmaf(__uint_as_float(u[i] << 16), x[2 * i], s);
      s = fmaf(__uint_as_float(u[i] & 0xFFFF0000u), x[2 * i + 1], s);
    }
    return s;
  } else {
    float s = 0.0f;
    s = fmaf(__uint_as_float(w.x), x[0], s);
    s = fmaf(__uint_as_float(w.y), x[1], s);
    s = fmaf(__uint_as_float(w.z), x[2], s);
    s = fmaf(__uint_as_float(w.w), x[3], s);
    return s;
  }
}

// VEC: rows are whole 16-byte pieces and 16-byte aligned; otherwise one
// element per lane step.
template <bool BF16, bool VEC>
__global__ __launch_bounds__(256) void k_dense_matvec(const void *__restrict__ w, const float *__restrict__ x,
                                                      float *__restrict__ y, int n, int k) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= n) return;  // whole waves leave together
  float acc = 0.0f;
  if constexpr (VEC) {
    constexpr int E = BF16 ? 8 : 4;  // elements per 16-byte piece
    const int pieces = k / E;
    const uint4 *wr = reinterpret_cast<const uint4 *>(static_cast<const uint8_t *>(w) + size_t(row) * k * (BF16 ? 2 : 4));
    int p = lane;
    for (; p + 64 < pieces; p += 128) {  // two pieces in flight
      const uint4 a = wr[p], b = wr[p + 64];
      float xa[E], xb[E];
#pragma unroll
      for (int i = 0; i < E; i += 4) {
        const float4 va = *reinterpret_cast<const float4 *>(x + p * E + i);
        const float4 vb = *reinterpret_cast<const float4 *>(x + (p + 64) * E + i);
        xa[i] = va.x, xa[i + 1] = va.y, xa[i + 2] = va.z, xa[i + 3] = va.w;
        xb[i] = vb.x, xb[i + 1] = vb.y, xb[i + 2] = vb.z, xb[i + 3] = vb.w;
      }
      acc += piece_dot<BF16>(a, xa);
      acc += piece_dot<BF16>(b, xb);
    }
    if (p < pieces) {
      const uint4 a = wr[p];
      float xa[E];
#pragma unroll
      for (int i = 0; i < E; i += 4) {
        const float4 va = *reinterpret_cast<const float4 *>(x + p * E + i);
        xa[i] = va.x, xa[i + 1] = va.y, xa[i + 2] = va.z, xa[i + 3] = va.w;
      }
      acc += piece_dot<BF16>(a, xa);
    }
  } else {
    for (int j = lane; j < k; j += 64) {
      const float wv = BF16 ? bf16_to_f32(static_cast<const uint16_t *>(w)[size_t(row) * k + j])
                            : static_cast<const float *>(w)[size_t(row) * k + j];
      acc = fmaf(wv, x[j], acc);
    }
  }
  acc = dev::wave_sum_xor(acc);
  if (lane == 0) y[row] = acc;
}

// Weights j..j+7 of a row (16-byte aligned): one 16-byte piece of bf16, two
// of fp32.
template <bool BF16>
__device__ __forceinline__ void load8(const uint8_t *row, int j, float (&v)[8]) {
  if constexpr (BF16) {
    const uint4 p = *reinterpret_cast<const uint4 *>(row + size_t(j) * 2);
    const uint32_t u[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(u[i] << 16);
      v[2 * i + 1] = __uint_as_float(u[i] & 0xFFFF0000u);
    }
  } else {
    const float4 a = *reinterpret_cast<const float4 *>(row + size_t(j) * 4);
    const float4 b = *reinterpret_cast<const float4 *>(row + size_t(j) * 4 + 16);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
  }
}
template <bool BF16>
__device__ __forceinline__ float weight_at(const void *w, size_t i) {
  return BF16 ? bf16_to_f32(static_cast<const uint16_t *>(w)[i]) : static_cast<const float *>(w)[i];
}

// Fused gate/up SwiGLU over F32 / BF16 weights, one row (TrySwiGLUVector's
// op 66, tensor.comp:38-48): h[r] = silu(Wg[r] . x) * (Wu[r] . x), the two
// rows read in one pass over x.  Gate and up may differ in type.  One wave
// per output row; VEC: rows are whole 8-element pieces, 16-byte aligned.
template <bool BG, bool BU, bool VEC>
__global__ __launch_bounds__(256) void k_dense_swiglu(const void *__restrict__ wg, const void *__restrict__ wu,
                                                      const float *__restrict__ x, float *__restrict__ y, int n,
                                                      int k) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= n) return;  // whole waves leave together
  float g = 0.0f, u = 0.0f;
  if constexpr (VEC) {
    const uint8_t *rg = static_cast<const uint8_t *>(wg) + size_t(row) * k * (BG ? 2 : 4);
    const uint8_t *ru = static_cast<const uint8_t *>(wu) + size_t(row) * k * (BU ? 2 : 4);
    for (int j = lane * 8; j < k; j += 512) {
      float a[8], b[8], xv[8];
      load8<BG>(rg, j, a);
      load8<BU>(ru, j, b);
      const float4 x0 = *reinterpret_cast<const float4 *>(x + j), x1 = *reinterpret_cast<const float4 *>(x + j + 4);
      xv[0] = x0.x, xv[1] = x0.y, xv[2] = x0.z, xv[3] = x0.w, xv[4] = x1.x, xv[5] = x1.y, xv[6] = x1.z, xv[7] = x1.w;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        g = fmaf(a[i], xv[i], g);
        u = fmaf(b[i], xv[i], u);
      }
    }
  } else {
    for (int j = lane; j < k; j += 64) {
      const float xv = x[j];
      g = fmaf(weight_at<BG>(wg, size_t(row) * k + j), xv, g);
      u = fmaf(weight_at<BU>(wu, size_t(row) * k + j), xv, u);
    }
  }
  g = dev::wave_sum_xor(g);
  u = dev::wave_sum_xor(u);
  if (lane == 0) {
    const float sg = g >= 20.0f ? g : (g <= -20.0f ? 0.0f : g / (1.0f + expf(-g)));  // tensor.comp:22
    y[row] = sg * u;
  }
}

// ---- several rows: fp32 matrix cores ------------------------------------------
// Y[m][n] = sum_k X[m][k] W[n][k] on v_mfma_f32_16x16x4_f32: fp32 products
// and sums, as the VALU's, at twice its rate and with no LDS staging.  Lane l
// of a wave holds elements 8q .. 8q+7 (q = l / 16) of a 32-element K-step of
// row l % 16 of X and of W, and MFMA i of the step takes element i of both:
// the same permutation of k on both sides.  A wave computes 16 TM x 16 TN of
// Y, and the KW waves of a workgroup take the K-steps in turn, requesting the
// next step's pieces before the current step's products, and meet in LDS in
// wave order.  The work is small and its chain long (the router: 128 x 128
// outputs over 2048 elements), so what bounds it is the latency of a wave's
// few loads: small outputs take 16 waves per 16 x 16 tile (64 workgroups of 4
// steps per wave at the router's shape), larger ones 32 x 32 tiles, where a
// loaded piece feeds two products, with fewer waves per tile.
// Measured (kernel trace, bf16 router of 128 experts, 128 rows of 2048): a
// tile of 64 x 16 outputs per workgroup with LDS-staged scalar products took
// 189.6 us (16 workgroups, 64 barriers), this 7.6 us.
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <bool BF16, bool VEC>
__device__ __forceinline__ void load_step(float (&v)[8], const void *base, size_t row, int k, int j) {
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = 0.0f;
  if constexpr (VEC) {  // k % 8 == 0: the lane's 8 elements are all inside the row or all past it
    if (j < k) load8<BF16>(static_cast<const uint8_t *>(base) + row * size_t(k) * (BF16 ? 2 : 4), j, v);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (j + i < k) v[i] = weight_at<BF16>(base, row * size_t(k) + j + i);
  }
}

template <bool BF16, bool VEC, int TM, int TN, int KW>
__global__ __launch_bounds__(64 * KW) void k_dense_mm(const void *__restrict__ w, const float *__restrict__ x,
                                                      float *__restrict__ y, int m, int n, int k) {
  __shared__ float red[KW][TM * TN * 4][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const int n0 = blockIdx.x * 16 * TN, m0 = blockIdx.y * 16 * TM;
  size_t xr[TM], wr[TN];  // rows past the end read the last one; their outputs are not written
#pragma unroll
  for (int i = 0; i < TM; ++i) xr[i] = size_t(min(m0 + 16 * i + r, m - 1));
#pragma unroll
  for (int i = 0; i < TN; ++i) wr[i] = size_t(min(n0 + 16 * i + r, n - 1));
  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float xa[2][TM][8], wa[2][TN][8];
  auto load = [&](int s, int k0) {
#pragma unroll
    for (int i = 0; i < TM; ++i) load_step<false, VEC>(xa[s][i], x, xr[i], k, k0 + 8 * q);
#pragma unroll
    for (int i = 0; i < TN; ++i) load_step<BF16, VEC>(wa[s][i], w, wr[i], k, k0 + 8 * q);
  };
  auto products = [&](int s) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[s][i][e], wa[s][j][e], acc[i][j], 0, 0, 0);
  };
  int k0 = wave * 32;
  if (k0 < k) load(0, k0);
  for (; k0 < k; k0 += 64 * KW) {  // two steps per turn, so that the stages are indexed statically
    const int k1 = k0 + 32 * KW, k2 = k0 + 64 * KW;
    if (k1 < k) load(1, k1);
    products(0);
    if (k2 < k) load(0, k2);
    if (k1 < k) products(1);
  }
  // Lane l holds rows 4q .. 4q+3 of column r of each 16 x 16 tile.
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) red[wave][(i * TN + j) * 4 + e][lane] = acc[i][j][e];
  __syncthreads();
  for (int o = wave; o < TM * TN * 4; o += KW) {
    float v = 0.0f;
#pragma unroll
    for (int p = 0; p < KW; ++p) v += red[p][o][lane];
    const int tile = o >> 2, row = m0 + 16 * (tile / TN) + 4 * q + (o & 3), col = n0 + 16 * (tile % TN) + r;
    if (row < m && col < n) y[size_t(row) * n + col] = v;
  }
}

}  // namespace

void dense_matvec_launch(const void *w, int bf16, const float *x, float *y, int n, int k, hipStream_t s) {
  const int es = bf16 ? 2 : 4;
  const bool vec = (size_t(k) * es) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(x) % 16 == 0;
  const dim3 grid((n + 3) / 4), block(256);
  if (bf16) {
    if (vec) hipLaunchKernelGGL((k_dense_matvec<true, true>), grid, block, 0, s, w, x, y, n, k);
    else hipLaunchKernelGGL((k_dense_matvec<true, false>), grid, block, 0, s, w, x, y, n, k);
  } else {
    if (vec) hipLaunchKernelGGL((k_dense_matvec<false, true>), grid, block, 0, s, w, x, y, n, k);
    else hipLaunchKernelGGL((k_dense_matvec<false, false>), grid, block, 0, s, w, x, y, n, k);
  }
  hip_check(hipGetLastError(), "dense matvec launch");
}

void dense_swiglu_launch(const void *wg, int bg, const void *wu, int bu, const float *x, float *y, int n, int k,
                         hipStream_t s) {
  const bool vec = k % 8 == 0 && reinterpret_cast<uintptr_t>(wg) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(wu) % 16 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0;
  const dim3 grid((n + 3) / 4), block(256);
#define QNN_SWIGLU_CASE(G, U)                                                                     \
  if (bool(bg) == G && bool(bu) == U) {                                                          \
    if (vec) hipLaunchKernelGGL((k_dense_swiglu<G, U, true>), grid, block, 0, s, wg, wu, x, y, n, k); \
    else hipLaunchKernelGGL((k_dense_swiglu<G, U, false>), grid, block, 0, s, wg, wu, x, y, n, k);    \
  }
  QNN_SWIGLU_CASE(false, false)
  QNN_SWIGLU_CASE(false, true)
  QNN_SWIGLU_CASE(true, false)
  QNN_SWIGLU_CASE(true, true)
#undef QNN_SWIGLU_CASE
  hip_check(hipGetLastError(), "dense swiglu launch");
}

void dense_gemm_launch(const void *w, int bf16, const float *x, float *y, int m, int n, int k, hipStream_t s) {
  // 16-byte pieces of both operands: whole 8-element chunks, aligned rows.
  const bool vec = k % 8 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0;
  // 32 x 32 tiles where they still give a workgroup for every second CU, with
  // more waves per tile while there are fewer than two per CU.
  auto tiles = [&](int t) { return (long long)((m + t - 1) / t) * ((n + t - 1) / t); };
#define QNN_DENSE_MM(TM, TN, KW)                                                                              \
  do {                                                                                                        \
    const dim3 grid((n + 16 * TN - 1) / (16 * TN), (m + 16 * TM - 1) / (16 * TM)), block(64 * KW);            \
    if (bf16) {                                                                                               \
      if (vec) hipLaunchKernelGGL((k_dense_mm<true, true, TM, TN, KW>), grid, block, 0, s, w, x, y, m, n, k); \
      else hipLaunchKernelGGL((k_dense_mm<true, false, TM, TN, KW>), grid, block, 0, s, w, x, y, m, n, k);    \
    } else {                                                                                                  \
      if (vec) hipLaunchKernelGGL((k_dense_mm<false, true, TM, TN, KW>), grid, block, 0, s, w, x, y, m, n, k); \
      else hipLaunchKernelGGL((k_dense_mm<false, false, TM, TN, KW>), grid, block, 0, s, w, x, y, m, n, k);   \
    }                                                                                                         \
  } while (0)
  if (tiles(32) >= 512) QNN_DENSE_MM(2, 2, 4);
  else if (tiles(32) >= 128) QNN_DENSE_MM(2, 2, 8);
  else QNN_DENSE_MM(1, 1, 16);
#undef QNN_DENSE_MM
  hip_check(hipGetLastError(), "dense gemm launch");
}

}  // namespace qnn
