// qnn_attention_mm.hip -- cached attention of many query rows (prompt chunks)
// on the fp16 matrix cores.
//
// k_attn (qnn_decode.hip) gives every query row its own workgroups, each of
// which reads its chunk of K and V and multiplies on the VALU: 128 rows over
// 4096 keys read the cache 128 times (460 us).  Here a workgroup holds 128
// query rows of one KV head (the query heads of the group are rows too) and
// walks a range of keys once, in tiles of KT.
//
// Both products take fp32 operands as two fp16 planes, hi = fp16(v), lo =
// fp16(v - hi), and run hi hi + lo hi + hi lo on v_mfma_f32_32x32x16_f16 with
// fp32 accumulation; scores, softmax, running maxima and sums are fp32.  hi and
// lo hold a value to 2^-24 of itself, as long as lo is a normal fp16 number:
// down to 2^-15 or so of the largest that shares its scale, below that to 2^-38
// of that largest.  So what has a scale of its own is small: every key's K and
// V (a score is one key's, and a key's V scale goes into its weight), every
// query row, and every row's weights w = p 2^(V's exponent), by the largest w
// of the row so far.  A key that a row does not see, by the mask, a later
// position or the window, has w = 0 there, and whatever finite values it holds
// reach nothing else; with one scale for a tile's keys a hidden value of 1e8
// times the others cost the result 1e-4, of 1e12 all of it.
//
// Layout.  S^T = K Q^T, so a lane's results are keys of ONE query row (column
// l % 32): maxima and sums are in-lane but for one exchange of the two
// half-waves, the rescale factor of the output is one register, and registers
// 8s .. 8s+7 of a score tile are, as they stand, the B operand (16 keys x 32
// rows) of K-step s of O^T = V^T P^T, with V's pieces written in the same key
// order.  The fragments of a tile are written to LDS by the workgroup (each
// thread turns 4 x 8 elements: K comes transposed, channels x keys, V as keys
// x channels) and read by its four waves, 32 query rows each; the next tile's
// elements are on their way to registers meanwhile.
//
// What bounds it: the VALU (softmax, planes of w, a share of the planes of K and
// V).  Counters, 128 rows over 4096 keys: 17 VALU operations per MFMA, so per 64
// keys and wave 1640 of 4 cycles against 96 MFMAs of 32, which two waves per
// SIMD run under each other's products; VALU busy 49 % and matrix cores 19 % of
// the elapsed cycles, waves waiting 26 % of theirs.  At dim 128
// that takes tiles of 32 keys (236 registers; 64 keys do not fit two waves per
// SIMD).  A KV head's keys are split over two workgroups per CU; k_attn_merge
// joins the parts.  Infinities and NaNs among a workgroup's keys or query rows
// send its part to a plain fp32 loop over its rows, four per wave, since 0 times
// them would reach rows that do not see the key, and NaN where the score is
// infinite.  (128 rows over 4096 keys with one hidden NaN: 1.05 ms, a row per
// wave and a key at a time 5.4; k_attn 0.46.)
// More than 128 channels stay with k_attn: at 256 the output of 32 rows (128
// registers) and the planes of q (128) are all that a wave of two per SIMD has.
//
// Measured (rotary, append and attention; 32 query heads on 8, dim 128), 128
// rows over 4096 keys 453 -> 63 us, over 16384 keys 1900 -> 160, 64 rows 224 ->
// 48, 16 rows 72 -> 31, 8 rows 45 -> 30 us (scales per tile and not per key: 1 to
// 3 us less, all in the two larger).  One against two workgroups per CU: 69
// against 65 us, 192 against 160 (four: 170).  Error against 64 bits 5.9e-7 ->
// 3.4e-7; over 60 drawn shapes that come here 0.74 to 0.84 of k_attn's.
// From when (attn_mm_plan): four rows, and rows x heads x keys of 512 k: 4
// rows of 32 heads over 4096 keys 31.2 -> 29.1 us, 2 rows 27.1 -> 30.6 (over
// 16384 keys 49.3 -> 63.2); 32 rows of 16 heads over 512 keys 26.0 -> 29.9,
// 128 rows 41.2 -> 32.9.  With 65 to 96 channels 640 k: 58 rows of 8 heads on
// 4, dim 80, soft cap, over 1207 keys (547 k) 32.6 -> 36.9; 107 rows of 8 on 2
// over 1097 (917 k) 39.3 -> 30.6.
// Soft cap: tanhf and a division by the cap took as long as all else on the
// VALU; tanh20 and a product: 20 rows of 28 heads on 4 over 2794 keys 40.3 ->
// 36.5 us, 102 rows of 8 on 4 over 765 keys, dim 64, 32.4 -> 28.4; error against
// 64 bits 3.34e-7 -> 3.38e-7.
#include "qnn_internal.h"
#include "qnn_lanes.h"

namespace qnn {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kQRows = 128;  // query rows (of one KV head) per workgroup, 32 per wave
constexpr uint32_t kInfBits = 0x7F800000u;

struct AttnMmArgs {
  const float *q, *cache;
  float *out, *opart, *ml;
  int rows, cap, heads, kv_heads, dim, position, window, masked, splits, qtiles, group;
  float softcap, scale;
};

__device__ __forceinline__ uint32_t abs_bits(float v) { return __float_as_uint(v) & 0x7FFFFFFFu; }
// A power of two for the planes of a row or key from its largest magnitude's
// bits: its exponent field, 2^-112 at least.  plane_scale brings the magnitude
// into [2^14, 2^15); plane_exp is the exponent that undoes it.
__device__ __forceinline__ uint32_t exp_field(uint32_t maxbits) { return max(maxbits & kInfBits, 15u << 23); }
__device__ __forceinline__ float plane_scale(uint32_t field) { return __uint_as_float((268u << 23) - field); }
__device__ __forceinline__ int plane_exp(uint32_t field) { return int(field >> 23) - 141; }

// Two fp16 planes of eight finite values, each times its power of two.
__device__ __forceinline__ void planes8(const float (&x)[8], const float (&scale)[8], uint4 &ph, uint4 &pl) {
  float hi[8], lo[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float s = x[i] * scale[i];
    hi[i] = float(_Float16(s));
    lo[i] = s - hi[i];
  }
  ph = make_uint4(pack_h2(hi[0], hi[1]), pack_h2(hi[2], hi[3]), pack_h2(hi[4], hi[5]), pack_h2(hi[6], hi[7]));
  pl = make_uint4(pack_h2(lo[0], lo[1]), pack_h2(lo[2], lo[3]), pack_h2(lo[4], lo[5]), pack_h2(lo[6], lo[7]));
}
__device__ __forceinline__ void planes8(const float (&x)[8], float scale, uint4 &ph, uint4 &pl) {
  const float s[8] = {scale, scale, scale, scale, scale, scale, scale, scale};
  planes8(x, s, ph, pl);
}

// Largest values over pairs of lanes, sixteen or thirty-two apart, of two
// values at once: lanes with that bit clear get a's, the others b's.
__device__ __forceinline__ uint32_t max_halves(uint32_t a, uint32_t b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  return max(uint32_t(r[0]), uint32_t(r[1]));
}
__device__ __forceinline__ uint32_t max_rows(uint32_t a, uint32_t b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  return max(uint32_t(r[0]), uint32_t(r[1]));
}
// The same for lanes one or two apart.
template <int OFF>
__device__ __forceinline__ uint32_t max_near(uint32_t a, uint32_t b, bool upper) {
  return max(upper ? b : a, uint32_t(dev::xor_lanes_i<OFF>(int(upper ? a : b))));
}
// A key's largest magnitude of K: m of a lane's four keys over the lanes that
// hold its other dims (bits 4 and 5, with tiles of 32 keys 3 too).  The lane
// keeps key lane / 16.
template <int KT>
__device__ __forceinline__ uint32_t k_key_max(const uint32_t (&m)[4]) {
  uint32_t v = max_rows(max_halves(m[0], m[2]), max_halves(m[1], m[3]));
  if (KT == 32) v = max(v, uint32_t(dev::xor_lanes_i<8>(int(v))));
  return v;
}
// A key's largest magnitude of V: m of a lane's eight keys over the lanes that
// hold its other channels: bits 0-2 and 5, with tiles of 32 keys 4 too.  The
// lane keeps key v_kept.
template <int KT>
__device__ __forceinline__ uint32_t v_key_max(const uint32_t (&m)[8], int lane) {
  constexpr int N = KT == 32 ? 2 : 4;
  uint32_t v[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    v[i] = KT == 32 ? max_rows(max_halves(m[i], m[4 + i]), max_halves(m[2 + i], m[6 + i])) : max_halves(m[i], m[4 + i]);
    v[i] = max(v[i], uint32_t(__builtin_amdgcn_mov_dpp(int(v[i]), 0x141, 0xF, 0xF, false)));  // lane 7 - l of its eight
  }
#pragma unroll
  for (int i = 0; i < N / 2; ++i) v[i] = max_near<1>(v[2 * i], v[2 * i + 1], lane & 1);
  if (KT == 32) return max(v[0], uint32_t(dev::xor_lanes_i<2>(int(v[0]))));
  return max_near<2>(v[0], v[1], lane & 2);
}
template <int KT>
__device__ __forceinline__ int v_kept(int lane) {
  return (lane & 1) + (KT == 32 ? lane >> 3 & 2 : lane & 2) + (lane >> 3 & 4);
}

__device__ __forceinline__ half8 as_half8(const uint4 &v) {
  half8 h;
  __builtin_memcpy(&h, &v, 16);
  return h;
}

// tanh for |x| <= 20: below 0.6 x + x^3 P(x^2), P fitted by least squares at
// Chebyshev nodes (4e-9 relative), above 1 - 2 / (e^2|x| + 1).  Within 1.7e-7
// of the value, as tanhf is (2 ulp), in 14 operations and no branch.
__device__ __forceinline__ float tanh20(float x) {
  const float a = fabsf(x), z = x * x;
  float p = fmaf(-0.00597367529f, z, 0.0208660811f);
  p = fmaf(p, z, -0.053805545f);
  p = fmaf(p, z, 0.133321926f);
  p = fmaf(p, z, -0.333333075f);
  const float small = fmaf(a * z, p, a);
  const float large = fmaf(-2.0f, __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(a * 2.88539008f) + 1.0f), 1.0f);
  return copysignf(a < 0.6f ? small : large, x);
}

typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc rsrc(const void *base, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, int(uint32_t(min(bytes, size_t(0xFFFFFFFFu)))),
                                           0x00020000);
}
// Four floats (any 4-byte alignment); zeros past the end of the buffer.  The
// whole offset is the lane's: a scalar offset need not take part in the check.
__device__ __forceinline__ float4 ld4(Rsrc r, uint32_t off) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, int(off), 0, 0);
  return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
}

// DP: head dimension padded to a multiple of 32; KT: keys per tile.  Waves 0
// and 1 hold a tile's K, thread x of them 4 keys from 4 (x % (KT / 4)) by 8 dims
// from 8 (x / (KT / 4)); waves 2 and 3 its V, thread x 8 keys by 4 channels.
template <int DP, int KT>
struct AttnMm {
  static constexpr int DS = DP / 16, CB = DP / 32, KB = KT / 32, KS = KT / 16;
  static constexpr int KF = KB * DS * 64, VF = CB * KS * 64;  // 16-byte pieces per plane
  static constexpr size_t lds = size_t(2 * KF + 2 * VF) * 16;
  static constexpr bool SPARE = KT * DP < 32 * 128;  // the last threads of both have dims, channels past DP
  static_assert(KT * DP <= 32 * 128, "a tile is 128 threads of 4 x 8 elements");
  // V: the channels from 4 v_group, the keys 16 (kk / 2) + 4 (kk % 2) + 0..3 and
  // 8..11.  Eight lanes read 128 bytes of a key; what else of a key the wave
  // holds lies in upper lanes (v_key_max).
  static __device__ __forceinline__ int v_group(int x) { return (x & 7) + (KT == 32 ? x >> 1 & 24 : x >> 2 & 8); }
  static __device__ __forceinline__ int v_kk(int x) {
    return KT == 32 ? (x >> 3 & 1) + (x >> 5 & 2) : (x >> 3 & 3) + (x >> 4 & 4);
  }
};

// EXTRA: a key mask or a soft cap.
template <int DP, int KT, bool EXTRA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_attn_mm(const AttnMmArgs a) {
  using T = AttnMm<DP, KT>;
  extern __shared__ uint4 lds[];
  uint4 *kf = lds, *vf = lds + 2 * T::KF;  // [plane][key block][dim step][lane], [plane][channel block][key step][lane]
  __shared__ __align__(16) uint32_t kmx[2][KT], vmx[KT];  // the tile's keys' largest magnitudes of K (per wave), V
  __shared__ __align__(16) int kex[KT];                   // exponents of their K planes
  __shared__ __align__(16) float vpw[KT];                 // powers of two of their V
  __shared__ __align__(16) uint32_t bad[4];               // per wave: an infinity or NaN
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int p = lane & 31, h = lane >> 5;
  // KV head fastest: with eight of them each XCD (as workgroups are usually
  // dealt) reads one head's keys.
  const int kh = blockIdx.x % a.kv_heads, rest = blockIdx.x / a.kv_heads;
  const int qt = rest % a.qtiles, split = rest / a.qtiles;
  const int nq = a.rows * a.group;                       // query rows of this KV head
  const int q0 = qt * kQRows, qi = q0 + wave * 32 + p;   // this lane's query row: row qi / group, head qi % group
  const bool qin = qi < nq;
  const int r = min(qi, nq - 1) / a.group, head = kh * a.group + min(qi, nq - 1) % a.group;
  const size_t width = size_t(a.kv_heads) * a.dim;
  const float *kt = a.cache + size_t(kh) * a.dim * a.cap;
  const float *vb = a.cache + size_t(a.cap) * width + size_t(kh) * a.cap * a.dim;
  const unsigned *mask =
      reinterpret_cast<const unsigned *>(a.cache + 2 * size_t(a.cap) * width) + size_t(r) * a.cap;
  const bool cvec = (a.dim & 3) == 0;

  // Keys of this lane's row, of its wave's rows (all of them, and those every
  // row has) and of the workgroup's.
  auto first_key = [&](int row) { return a.window > 0 && a.position + row + 1 > a.window ? a.position + row + 1 - a.window : 0; };
  const int kbeg = first_key(r), kend = a.position + r + 1;
  const int w0 = min(q0 + wave * 32, nq - 1) / a.group, w1 = min(q0 + wave * 32 + 31, nq - 1) / a.group;
  const int both0 = first_key(w1), both1 = a.position + w0 + 1;
  const int g0 = q0 / a.group, g1 = min(q0 + kQRows - 1, nq - 1) / a.group;
  const int klo = first_key(g0), khi = a.position + g1 + 1;
  const int t0 = klo / KT, nt = (khi + KT - 1) / KT - t0;
  const int tb = t0 + int((long long)nt * split / a.splits), te = t0 + int((long long)nt * (split + 1) / a.splits);
  const bool busy = q0 + wave * 32 < nq;  // waves past the last query row only prepare keys

  // ---- this lane's query row as B fragments: dims 16 ds + 8 h .. + 7
  half8 qh[T::DS], ql[T::DS];
  int qexp;  // exponent of a score, but for the key's
  bool qbad = false;  // an infinity or NaN in this wave's query rows: 0 times it would be in the planes' products
  {
    float qv[T::DS][8];
    // The score's scale as a factor in [0.5, 1), taken into q, and an exponent.
    int sexp;
    const float sfac = frexpf(a.scale > 0.0f ? a.scale : 1.0f / sqrtf(float(a.dim)), &sexp);
    const float *qr = a.q + (size_t(r) * a.heads + head) * a.dim;
    uint32_t mx = 0;
#pragma unroll
    for (int ds = 0; ds < T::DS; ++ds) {
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        const int d = 16 * ds + 8 * h + e;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (cvec) {
          if (d < a.dim) v = *reinterpret_cast<const float4 *>(qr + d);
        } else {
          if (d < a.dim) v.x = qr[d];
          if (d + 1 < a.dim) v.y = qr[d + 1];
          if (d + 2 < a.dim) v.z = qr[d + 2];
          if (d + 3 < a.dim) v.w = qr[d + 3];
        }
        qv[ds][e] = v.x, qv[ds][e + 1] = v.y, qv[ds][e + 2] = v.z, qv[ds][e + 3] = v.w;
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        qv[ds][e] *= sfac;
        mx = max(mx, abs_bits(qv[ds][e]));
      }
    }
    qbad = __ballot(mx >= kInfBits) != 0;
    mx = max(mx, uint32_t(dev::xor_lanes_i<32>(int(mx))));
    const uint32_t ef = exp_field(mx);
    const float s = plane_scale(ef);
#pragma unroll
    for (int ds = 0; ds < T::DS; ++ds) {
      uint4 ph, pl;
      planes8(qv[ds], s, ph, pl);
      qh[ds] = as_half8(ph);
      ql[ds] = as_half8(pl);
    }
    qexp = plane_exp(ef) + sexp;
  }

  // ---- this thread's share of a tile
  float4 raw[8];  // K: dim e of the four keys; V: key e's four channels
  const bool isk = wave < 2;  // uniform
  const int x = tid & 127;
  const int kkey = 4 * (x % (KT / 4)), kdim = 8 * (x / (KT / 4));
  const int vch = 4 * T::v_group(x), vkey = 16 * (T::v_kk(x) >> 1) + 4 * (T::v_kk(x) & 1);
  const bool spare = T::SPARE && (isk ? kdim : vch) >= DP;  // nothing to hold, whatever was loaded
  // Buffer loads: dims past the last and keys past the capacity read zeros or
  // other elements of the head.  Keys outside the workgroup's range and
  // channels past the last are zeroed after the load.
  const Rsrc krs = rsrc(kt, size_t(a.dim) * a.cap * 4), vrs = rsrc(vb, size_t(a.cap) * a.dim * 4);
  const uint32_t off0 = (isk ? uint32_t(kdim) * uint32_t(a.cap) + uint32_t(kkey) : uint32_t(vkey) * uint32_t(a.dim) + uint32_t(vch)) * 4u;
  auto load_tile = [&](int t) {
    // (Opaque, or the eight rows' sums are kept in registers of their own.)
    uint32_t at = off0 + uint32_t(t) * KT * (isk ? 1u : uint32_t(a.dim)) * 4u;
    asm("" : "+v"(at));
    if (isk) {
#pragma unroll
      for (int e = 0; e < 8; ++e) raw[e] = ld4(krs, at + uint32_t(e) * uint32_t(a.cap) * 4u);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) raw[e] = ld4(vrs, at + (8u * (e >> 2) + (e & 3)) * uint32_t(a.dim) * 4u);
    }
  };
  auto trim_tile = [&](int t) {
    const int k0 = t * KT;
    const bool inside = k0 >= klo && k0 + KT <= khi;  // uniform
    if (inside && a.dim == DP) return;
    if (isk) {
      const int key = k0 + kkey;
      if (inside) return;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float4 &v = raw[e];
        v.x = key >= klo && key < khi ? v.x : 0.0f;
        v.y = key + 1 >= klo && key + 1 < khi ? v.y : 0.0f;
        v.z = key + 2 >= klo && key + 2 < khi ? v.z : 0.0f;
        v.w = key + 3 >= klo && key + 3 < khi ? v.w : 0.0f;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int key = k0 + vkey + 8 * (e >> 2) + (e & 3);
        const int n = key >= klo && key < khi ? a.dim - vch : 0;  // channels from vch
        float4 &v = raw[e];
        v.x = n > 0 ? v.x : 0.0f;
        v.y = n > 1 ? v.y : 0.0f;
        v.z = n > 2 ? v.z : 0.0f;
        v.w = n > 3 ? v.w : 0.0f;
      }
    }
  };
  // Every key's largest magnitudes, of K as far as this wave holds it.
  auto key_maxima = [&]() {
    uint32_t top;
    if (isk) {
      uint32_t m[4] = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        m[0] = max(m[0], abs_bits(raw[e].x));
        m[1] = max(m[1], abs_bits(raw[e].y));
        m[2] = max(m[2], abs_bits(raw[e].z));
        m[3] = max(m[3], abs_bits(raw[e].w));
      }
      top = k_key_max<KT>(m);
      kmx[wave & 1][kkey + (lane >> 4)] = top;
    } else {
      uint32_t m[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        m[e] = max(max(abs_bits(raw[e].x), abs_bits(raw[e].y)), max(abs_bits(raw[e].z), abs_bits(raw[e].w)));
        if (spare) m[e] = 0u;
      }
      top = v_key_max<KT>(m, lane);
      const int e = v_kept<KT>(lane);
      vmx[vkey + 8 * (e >> 2) + (e & 3)] = top;
    }
    const bool inf = qbad || __ballot(top >= kInfBits) != 0;
    if (lane == 0) bad[wave] = inf;
  };
  auto k_field4 = [&](int key) {
    const uint4 m = *reinterpret_cast<const uint4 *>(&kmx[0][key]), o = *reinterpret_cast<const uint4 *>(&kmx[1][key]);
    return make_uint4(exp_field(max(m.x, o.x)), exp_field(max(m.y, o.y)), exp_field(max(m.z, o.z)), exp_field(max(m.w, o.w)));
  };
  auto v_field4 = [&](int key) {
    const uint4 m = *reinterpret_cast<const uint4 *>(&vmx[key]);
    return make_uint4(exp_field(m.x), exp_field(m.y), exp_field(m.z), exp_field(m.w));
  };
  auto write_tile = [&]() {
    if (tid < KT / 4) {
      const uint4 k = k_field4(4 * tid), v = v_field4(4 * tid);
      *reinterpret_cast<int4 *>(&kex[4 * tid]) = make_int4(plane_exp(k.x), plane_exp(k.y), plane_exp(k.z), plane_exp(k.w));
      *reinterpret_cast<uint4 *>(&vpw[4 * tid]) = v;
    }
    uint4 *dst;
    int plane;
    float sk[4], sv[8];  // plane scales of the keys
    if (isk) {
      dst = kf + ((kkey >> 5) * T::DS + (kdim >> 4)) * 64 + (kkey & 31) + 4 * (kdim & 8);
      plane = T::KF;
      const uint4 f = k_field4(kkey);
      sk[0] = plane_scale(f.x), sk[1] = plane_scale(f.y), sk[2] = plane_scale(f.z), sk[3] = plane_scale(f.w);
    } else {
      dst = vf + ((vch >> 5) * T::KS + (vkey >> 4)) * 64 + (vch & 31) + 8 * (vkey & 4);
      plane = T::VF;
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        const uint4 f = v_field4(vkey + 2 * e);
        sv[e] = plane_scale(f.x), sv[e + 1] = plane_scale(f.y), sv[e + 2] = plane_scale(f.z), sv[e + 3] = plane_scale(f.w);
      }
    }
    if (spare) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = i == 0 ? raw[e].x : (i == 1 ? raw[e].y : (i == 2 ? raw[e].z : raw[e].w));
      if (isk) planes8(v, sk[i], dst[i], dst[plane + i]);
      else planes8(v, sv, dst[i], dst[plane + i]);
    }
  };

  f32x16 acc[T::CB];
#pragma unroll
  for (int c = 0; c < T::CB; ++c)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[c][e] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;  // l_run: this half-wave's keys
  bool slow = false;
  // A row's weights of a tile's values are w = p 2^(the key's V exponent), in
  // planes of the row's own scale: by the largest w up to this tile, falling as
  // the running maximum of the scores leaves them behind.
  float w_run = 0.0f;  // acc holds O 2^28 / (its power of two, at least 2^-112)

  if (tb < te) load_tile(tb);
  for (int t = tb; t < te; ++t) {
    trim_tile(t);
    key_maxima();
    __syncthreads();  // the maxima, and every wave is done with the previous tile's fragments
    {
      const uint4 f = *reinterpret_cast<const uint4 *>(bad);
      if (f.x | f.y | f.z | f.w) {  // uniform: an infinity or NaN among the keys or in q
        slow = true;
        break;
      }
    }
    write_tile();
    if (t + 1 < te) load_tile(t + 1);
    __syncthreads();

    float s[T::KB][16];
    if (busy) {
      // ---- scores of this lane's row: keys 32 kb + 8 (i / 4) + 4 h + i % 4
      // (Fragments are read one step ahead of their products.)
      uint4 fh[2], fl[2];
      fh[0] = kf[lane];
      fl[0] = kf[T::KF + lane];
      f32x16 d = {};
#pragma unroll
      for (int n = 0; n < T::KB * T::DS; ++n) {
        const int kb = n / T::DS, ds = n % T::DS;
        if (n + 1 < T::KB * T::DS) {
          fh[(n + 1) & 1] = kf[(n + 1) * 64 + lane];
          fl[(n + 1) & 1] = kf[T::KF + (n + 1) * 64 + lane];
        }
        const half8 kh8 = as_half8(fh[n & 1]), kl8 = as_half8(fl[n & 1]);
        d = __builtin_amdgcn_mfma_f32_32x32x16_f16(kl8, qh[ds], d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh8, ql[ds], d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh8, qh[ds], d, 0, 0, 0);
        if (ds == T::DS - 1) {
#pragma unroll
          for (int i = 0; i < 16; i += 4) {
            const int4 ke = *reinterpret_cast<const int4 *>(&kex[32 * kb + 2 * i + 4 * h]);
            s[kb][i] = ldexpf(d[i], qexp + ke.x);
            s[kb][i + 1] = ldexpf(d[i + 1], qexp + ke.y);
            s[kb][i + 2] = ldexpf(d[i + 2], qexp + ke.z);
            s[kb][i + 3] = ldexpf(d[i + 3], qexp + ke.w);
          }
          d = f32x16{};
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (EXTRA && a.softcap > 0.0f) {
        const float inv = 1.0f / a.softcap;
#pragma unroll
        for (int kb = 0; kb < T::KB; ++kb)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            s[kb][i] = a.softcap * tanh20(fminf(fmaxf(s[kb][i] * inv, -20.0f), 20.0f));
      }
      const int k0 = t * KT;
      const bool valid_all = k0 >= both0 && k0 + KT <= both1 && !(EXTRA && a.masked);  // uniform
      if (!valid_all) {
#pragma unroll
        for (int kb = 0; kb < T::KB; ++kb)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int key = k0 + 32 * kb + 8 * (i >> 2) + 4 * h + (i & 3);
            bool ok = key >= kbeg && key < kend;
            if (EXTRA && ok && a.masked) ok = mask[key] != 0u;
            if (!ok) s[kb][i] = -INFINITY;
          }
      }
      // ---- online softmax
      float mx = s[0][0];
#pragma unroll
      for (int kb = 0; kb < T::KB; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[kb][i]);
      mx = fmaxf(mx, dev::xor_lanes<32>(mx));
      const float m_new = fmaxf(m_run, mx);
      const float m_sub = m_new == -INFINITY ? 0.0f : m_new;  // no key yet: every p is exp(-inf) = 0
      const float keep = __expf(m_run - m_sub);
      float sum = 0.0f, wmx = 0.0f;
#pragma unroll
      for (int kb = 0; kb < T::KB; ++kb)
#pragma unroll
        for (int i = 0; i < 16; i += 4) {
          const float4 vs = *reinterpret_cast<const float4 *>(&vpw[32 * kb + 2 * i + 4 * h]);
          const float ve[4] = {vs.x, vs.y, vs.z, vs.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float p = __expf(s[kb][i + e] - m_sub);
            sum += p;
            s[kb][i + e] = p * ve[e];
            wmx = fmaxf(wmx, s[kb][i + e]);
          }
        }
      l_run = l_run * keep + sum;
      m_run = m_new;
      wmx = fmaxf(wmx, dev::xor_lanes<32>(wmx));
      const uint32_t w_old = exp_field(__float_as_uint(w_run));
      w_run = fmaxf(w_run * keep, wmx);
      const uint32_t w_new = exp_field(__float_as_uint(w_run));
      const float wscale = plane_scale(w_new);
      // acc to the new maximum and the new scale (skipped when no row changes)
      const float f = ldexpf(keep, (int(w_old) - int(w_new)) >> 23);
      if (__ballot(f != 1.0f) != 0) {
#pragma unroll
        for (int c = 0; c < T::CB; ++c)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[c][e] *= f;
      }
      // ---- values
      half8 p_h[2], p_l[2];
      auto p_planes = [&](int ks) {
        float pv[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) pv[e] = s[ks >> 1][8 * (ks & 1) + e];
        uint4 ph, pl;
        planes8(pv, wscale, ph, pl);
        p_h[ks & 1] = as_half8(ph);
        p_l[ks & 1] = as_half8(pl);
      };
      // Step n: channel block n % CB of key step n / CB.
      auto v_at = [&](int n) { return ((n % T::CB) * T::KS + n / T::CB) * 64 + lane; };
      p_planes(0);
      fh[0] = vf[v_at(0)];
      fl[0] = vf[T::VF + v_at(0)];
#pragma unroll
      for (int n = 0; n < T::CB * T::KS; ++n) {
        const int ks = n / T::CB, c = n % T::CB;
        if (n + 1 < T::CB * T::KS) {
          fh[(n + 1) & 1] = vf[v_at(n + 1)];
          fl[(n + 1) & 1] = vf[T::VF + v_at(n + 1)];
        }
        const half8 vh = as_half8(fh[n & 1]), vl = as_half8(fl[n & 1]);
        acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, p_h[ks & 1], acc[c], 0, 0, 0);
        acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, p_l[ks & 1], acc[c], 0, 0, 0);
        acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, p_h[ks & 1], acc[c], 0, 0, 0);
        if (c == 0 && ks + 1 < T::KS) p_planes(ks + 1);  // in these products' shadow
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  if (slow) {
    // Infinities or NaNs among the keys would reach rows that do not see them
    // through the products' zeros, and in q would meet the zeros of the lower
    // planes (inf, which a soft cap makes finite, would be NaN): this part is
    // computed in fp32 as k_attn does, a wave per four query rows: a lane per key
    // for the scores, per channel for the values.
    constexpr int R = 4;
    const float mul = a.scale > 0.0f ? a.scale : 1.0f / sqrtf(float(a.dim));
    const unsigned *m0 = reinterpret_cast<const unsigned *>(a.cache + 2 * size_t(a.cap) * width);
    const int c0 = min(lane, a.dim - 1), c1 = min(lane + 64, a.dim - 1);
    for (int i = R * wave; i < kQRows && q0 + i < nq; i += 4 * R) {
      int row[R];
      size_t rh[R];
      float m[R], l[R], o[R][2];  // channels lane, lane + 64
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int x = min(q0 + i + j, nq - 1);
        row[j] = x / a.group;
        rh[j] = size_t(row[j]) * a.heads + kh * a.group + x % a.group;
        m[j] = -INFINITY;
        l[j] = o[j][0] = o[j][1] = 0.0f;
      }
      const int first = max(first_key(row[0]), tb * KT), end = min(a.position + row[R - 1] + 1, te * KT);
      for (int k0 = first; k0 < end; k0 += 64) {
        const int key = min(k0 + lane, end - 1);
        float d[R], w[R];
        uint64_t seen[R];
#pragma unroll
        for (int j = 0; j < R; ++j) d[j] = 0.0f;
#pragma unroll 8
        for (int c = 0; c < a.dim; ++c) {
          const float kv = kt[size_t(c) * a.cap + key];
#pragma unroll
          for (int j = 0; j < R; ++j) d[j] += a.q[rh[j] * a.dim + c] * kv;
        }
#pragma unroll
        for (int j = 0; j < R; ++j) {
          bool ok = k0 + lane < end && key >= first_key(row[j]) && key <= a.position + row[j];
          if (ok && a.masked) ok = m0[size_t(row[j]) * a.cap + key] != 0u;
          float sc = d[j] * mul;
          if (a.softcap > 0.0f) sc = a.softcap * tanhf(fminf(fmaxf(sc / a.softcap, -20.0f), 20.0f));
          const float mn = fmaxf(m[j], dev::wave_max_xor(ok ? sc : -INFINITY));
          const float kp = mn == -INFINITY ? 1.0f : expf(m[j] - mn);
          w[j] = ok && sc != -INFINITY ? expf(sc - mn) : 0.0f;  // (a NaN before any other key counts, too)
          l[j] = l[j] * kp + dev::wave_sum_xor(w[j]);
          m[j] = mn;
          o[j][0] *= kp;
          o[j][1] *= kp;
          seen[j] = __ballot(ok);
        }
        for (int u0 = 0; u0 < min(64, end - k0); u0 += 8) {
#pragma unroll
          for (int u = u0; u < u0 + 8; ++u) {
            const float *v = vb + size_t(min(k0 + u, end - 1)) * a.dim;
            const float v0 = v[c0], v1 = v[c1];
#pragma unroll
            for (int j = 0; j < R; ++j) {
              const float wu = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w[j]), u));
              const bool see = (seen[j] >> u) & 1u;  // what the row does not see may be anything
              const float a0 = wu * v0, a1 = wu * v1;
              o[j][0] += see ? a0 : 0.0f;
              o[j][1] += see ? a1 : 0.0f;
            }
          }
        }
      }
#pragma unroll
      for (int j = 0; j < R; ++j) {
        if (q0 + i + j >= nq) continue;
        const bool whole = a.splits == 1;
        float *dst = whole ? a.out + rh[j] * a.dim : a.opart + (size_t(split) * a.rows * a.heads + rh[j]) * a.dim;
        if (lane < a.dim) dst[lane] = whole ? o[j][0] / l[j] : o[j][0];
        if (lane + 64 < a.dim) dst[lane + 64] = whole ? o[j][1] / l[j] : o[j][1];
        if (!whole && lane == 0) {
          float *ml = a.ml + (size_t(split) * a.rows * a.heads + rh[j]) * 2;
          ml[0] = m[j];
          ml[1] = l[j];
        }
      }
    }
    return;
  }

  if (!qin || !busy) return;
  const float l = l_run + dev::xor_lanes<32>(l_run);
  const int oexp = int(exp_field(__float_as_uint(w_run)) >> 23) - (127 + 28);
  const size_t row_head = size_t(r) * a.heads + head;
  const bool whole = a.splits == 1;
  float *o = whole ? a.out + row_head * a.dim : a.opart + (size_t(split) * a.rows * a.heads + row_head) * a.dim;
#pragma unroll
  for (int c = 0; c < T::CB; ++c)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int ch = 32 * c + 8 * g + 4 * h;
      if (ch >= a.dim) continue;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = ldexpf(acc[c][4 * g + e], oexp);
        if (whole) v[e] = v[e] / l;
      }
      if (cvec) {
        *reinterpret_cast<float4 *>(o + ch) = make_float4(v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (ch + e < a.dim) o[ch + e] = v[e];
      }
    }
  if (!whole && h == 0) {
    float *ml = a.ml + (size_t(split) * a.rows * a.heads + row_head) * 2;
    ml[0] = m_run;
    ml[1] = l;
  }
}

template <int DP, int KT, bool EXTRA>
void launch_as(const AttnMmArgs &a, hipStream_t s) {
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void *>(&k_attn_mm<DP, KT, EXTRA>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, int(AttnMm<DP, KT>::lds));
  hip_check(attr, "attention LDS size");
  k_attn_mm<DP, KT, EXTRA><<<a.kv_heads * a.qtiles * a.splits, 256, AttnMm<DP, KT>::lds, s>>>(a);
}
template <int DP, int KT>
void launch(const AttnMmArgs &a, hipStream_t s) {
  if (a.masked || a.softcap > 0.0f) launch_as<DP, KT, true>(a, s);
  else launch_as<DP, KT, false>(a, s);
}

}  // namespace

bool attn_mm_plan(AttnPlan &p, int rows, int cap, int heads, int kv_heads, int dim, int position, int window) {
  const int group = heads / kv_heads, min_k = tuning().attn_mm_min;
  const long long nq = (long long)rows * group;
  const int last_end = position + rows;
  const long long least = ((long long)min_k << 10) * (dim > 64 && dim <= 96 ? 5 : 4) / 4;
  if (min_k <= 0 || rows < 4 || dim > 128 || nq > (1 << 24) ||
      // 32-bit offsets within a KV head, those of dims past the last (up to 64 or 128) included
      size_t(dim) * cap * 4 > 0x7FFFFFFFull || size_t(dim <= 64 ? 64 : 128) * (size_t(cap) + 64) * 4 > 0xFFFFFFFFull ||
      (long long)rows * heads * (window > 0 ? std::min(window, last_end) : last_end) < least)
    return false;
  p.qtiles = int((nq + kQRows - 1) / kQRows);
  // The keys of one workgroup's rows: at most the window and those rows.
  const int longest = window > 0 ? int(std::min<long long>((long long)window + kQRows, last_end)) : last_end;
  const int tiles = (longest + 63) / 64;
  // Two workgroups per CU, at least two tiles of 64 keys (four of 32) each, and
  // four while there is a workgroup for every CU (shorter parts cost the merge
  // more than they save: 128 rows of 16 heads on 8, dim 96, over 3000 keys in 16
  // parts 42, in 23 45 us; 64 rows of 32 on 8, dim 128, over 4096 in 16 45.5, in 32 47.5).
  const long long wgs = (long long)kv_heads * p.qtiles, target = std::max(1, tuning().attn_wgs);
  const long long longer = std::max<long long>(tiles / 4, target / 2 / wgs);
  p.splits = int(std::max<long long>(1, std::min<long long>({target / wgs, tiles / 2, longer})));
  p.part_floats = p.splits > 1 ? size_t(p.splits) * rows * heads * (size_t(dim) + 2) : 0;
  return true;
}

void attn_mm_launch(const float *q, const float *cache, float *out, float *opart, float *ml, const AttnPlan &p, int rows,
                    int cap, int heads, int kv_heads, int dim, int position, int window, float softcap, float scale,
                    int masked, hipStream_t s) {
  AttnMmArgs a;
  a.q = q;
  a.cache = cache;
  a.out = out;
  a.opart = opart;
  a.ml = ml;
  a.rows = rows;
  a.cap = cap;
  a.heads = heads;
  a.kv_heads = kv_heads;
  a.dim = dim;
  a.position = position;
  a.window = window;
  a.masked = masked;
  a.splits = p.splits;
  a.qtiles = p.qtiles;
  a.group = heads / kv_heads;
  a.softcap = softcap;
  a.scale = scale;
  if (dim <= 64) launch<64, 64>(a, s);
  else if (dim <= 96) launch<96, 32>(a, s);
  else launch<128, 32>(a, s);
  hip_check(hipGetLastError(), "attention launch");
}

}  // namespace qnn
