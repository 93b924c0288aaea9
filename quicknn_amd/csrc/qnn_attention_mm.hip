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
// fp16(v - hi), 22 significant bits, and run hi hi + lo hi + hi lo on
// v_mfma_f32_32x32x16_f16 with fp32 accumulation; scores, softmax, running
// maxima and sums are fp32.  Powers of two keep the planes in fp16's range: q
// per row, K per tile, V by the largest of the tiles so far, p by 2^14 (each
// plane then resolves 2^-38 of the largest value it is scaled for).  The error
// against 64 bits is no larger than that of k_attn's fp32 sums.
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
// What bounds it: per 64 keys and wave 96 MFMAs (18.5 ns each) against about
// 1000 VALU operations (softmax, planes of p, a share of the planes of K and
// V), which two waves per SIMD run under each other's products.  At dim 128
// that takes tiles of 32 keys (221 registers; 64 keys take 343, one wave per
// SIMD).  A KV head's keys are split over two workgroups per CU; k_attn_merge
// joins the parts.  Infinities and NaNs among a workgroup's keys or query rows
// send its part to a plain loop over its rows, since 0 times them would reach
// rows that do not see the key, and NaN where the score is infinite.
//
// Measured (rotary, append and attention; 32 query heads on 8, dim 128), 128
// rows over 4096 keys 453 -> 64 us (64-key tiles 67), over 16384 keys 1914 ->
// 159 (190), 64 rows 232 -> 48, 16 rows 73 -> 33, 8 rows 45 -> 30 us; error
// against 64 bits 5.9e-7 -> 3.9e-7.  One against two workgroups per CU: 69
// against 64 us, 191 against 159; with four, 77 and 172.  At dim 96, where one
// fits a CU, 128 rows of 16 heads on 8 over 3000 keys: one 41, two 46 us.
// From when (attn_mm_plan): four rows, and rows x heads x keys of 512 k: 4
// rows of 32 heads over 4096 keys 32.2 -> 31.0 us, 2 rows 27.1 -> 30.6 (over
// 16384 keys 49.3 -> 63.2); 32 rows of 16 heads over 512 keys 26.6 -> 31.0,
// 128 rows 43.9 -> 34.6.  With 65 to 96 channels, one workgroup per CU, 640 k:
// 58 rows of 8 heads on 4, dim 80, soft cap, over 1207 keys (547 k) 33.3 ->
// 37.3; 107 rows of 8 on 2 over 1097 (917 k) 37.9 -> 28.9.
// Soft cap: tanhf and a division by the cap took as long as all else on the
// VALU; tanh20 and a product: 20 rows of 28 heads on 4 over 2794 keys 40.3 ->
// 36.5 us, 102 rows of 8 on 4 over 765 keys, dim 64, 32.4 -> 28.4 (k_attn:
// 213.6, 32.2); error against 64 bits 3.34e-7 -> 3.38e-7.
#include "qnn_internal.h"
#include "qnn_lanes.h"

namespace qnn {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kQRows = 128;  // query rows (of one KV head) per workgroup, 32 per wave
constexpr int kPExp = 14;    // p is held as p 2^14
constexpr uint32_t kInfBits = 0x7F800000u;

struct AttnMmArgs {
  const float *q, *cache;
  float *out, *opart, *ml;
  int rows, cap, heads, kv_heads, dim, position, window, masked, splits, qtiles, group;
  float softcap, scale;
};

__device__ __forceinline__ uint32_t abs_bits(float v) { return __float_as_uint(v) & 0x7FFFFFFFu; }
__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
  v = max(v, uint32_t(dev::xor_lanes_i<32>(int(v))));
  v = max(v, uint32_t(dev::xor_lanes_i<16>(int(v))));
  v = max(v, uint32_t(dev::xor_lanes_i<8>(int(v))));
  v = max(v, uint32_t(dev::xor_lanes_i<4>(int(v))));
  v = max(v, uint32_t(dev::xor_lanes_i<2>(int(v))));
  return max(v, uint32_t(dev::xor_lanes_i<1>(int(v))));
}
// Exponent for a largest finite magnitude; below 2^-110 (and for zeros, which
// ask for none) the scale stays 2^110, which is finite.
__device__ __forceinline__ int plane_exp(uint32_t maxbits) {
  return maxbits ? max(range_exp(__uint_as_float(maxbits)), -110) : -110;
}

// Two fp16 planes of eight finite values times a power of two.
__device__ __forceinline__ void planes8(const float (&x)[8], float scale, uint4 &ph, uint4 &pl) {
  float hi[8], lo[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float s = x[i] * scale;
    hi[i] = float(_Float16(s));
    lo[i] = s - hi[i];
  }
  ph = make_uint4(pack_h2(hi[0], hi[1]), pack_h2(hi[2], hi[3]), pack_h2(hi[4], hi[5]), pack_h2(hi[6], hi[7]));
  pl = make_uint4(pack_h2(lo[0], lo[1]), pack_h2(lo[2], lo[3]), pack_h2(lo[4], lo[5]), pack_h2(lo[6], lo[7]));
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

// DP: head dimension padded to a multiple of 32; KT: keys per tile.
template <int DP, int KT>
struct AttnMm {
  static constexpr int DS = DP / 16, CB = DP / 32, KB = KT / 32, KS = KT / 16;
  static constexpr int UK = KT * DP / 32;            // units of 4 x 8 elements of K, and as many of V
  static constexpr int NU = (2 * UK + 255) / 256;    // per thread
  static constexpr int KF = KB * DS * 64, VF = CB * KS * 64;  // 16-byte pieces per plane
  static constexpr size_t lds = size_t(2 * KF + 2 * VF) * 16;
  static_assert(UK % 64 == 0, "whole waves take K or V units");
};

// EXTRA: a key mask or a soft cap.
template <int DP, int KT, bool EXTRA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_attn_mm(const AttnMmArgs a) {
  using T = AttnMm<DP, KT>;
  extern __shared__ uint4 lds[];
  uint4 *kf = lds, *vf = lds + 2 * T::KF;  // [plane][key block][dim step][lane], [plane][channel block][key step][lane]
  __shared__ uint32_t red[2][2][4];        // [tile parity][K, V][wave]
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
  float qscale;  // score scale without the tile's exponent
  bool qbad = false;  // an infinity or NaN in this wave's query rows: 0 times it would be in the planes' products
  {
    float qv[T::DS][8];
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
      for (int e = 0; e < 8; ++e) mx = max(mx, abs_bits(qv[ds][e]));
    }
    qbad = __ballot(mx >= kInfBits) != 0;
    mx = max(mx, uint32_t(dev::xor_lanes_i<32>(int(mx))));
    const int e = plane_exp(mx);
    const float s = ldexpf(1.0f, -e);
#pragma unroll
    for (int ds = 0; ds < T::DS; ++ds) {
      uint4 ph, pl;
      planes8(qv[ds], s, ph, pl);
      qh[ds] = as_half8(ph);
      ql[ds] = as_half8(pl);
    }
    qscale = ldexpf(a.scale > 0.0f ? a.scale : 1.0f / sqrtf(float(a.dim)), e);
  }

  // ---- tile loads: unit u < UK is 4 keys x 8 dims of K, else 4 channels x 8 keys of V
  float4 raw[T::NU][8];
  auto unit_of = [&](int j) { return __builtin_amdgcn_readfirstlane((tid & ~63) + 256 * j) + lane; };
  // Buffer loads: dims past the last and keys past the capacity read zeros or
  // other elements of the head.  Keys outside the workgroup's range and
  // channels past the last are zeroed after the load.
  const Rsrc krs = rsrc(kt, size_t(a.dim) * a.cap * 4), vrs = rsrc(vb, size_t(a.cap) * a.dim * 4);
  uint32_t uoff[T::NU];
#pragma unroll
  for (int j = 0; j < T::NU; ++j) {
    const int u = unit_of(j);
    if (u - lane < T::UK) {
      uoff[j] = (uint32_t(8 * (u / (KT / 4))) * uint32_t(a.cap) + uint32_t(4 * (u % (KT / 4)))) * 4u;
    } else {
      const int x = u - T::UK, kk = x / (DP / 4);
      uoff[j] = (uint32_t(16 * (kk >> 1) + 4 * (kk & 1)) * uint32_t(a.dim) + uint32_t(4 * (x % (DP / 4)))) * 4u;
    }
  }
  auto load_tile = [&](int t) {
    const uint32_t k0 = uint32_t(t) * KT;
#pragma unroll
    for (int j = 0; j < T::NU; ++j) {
      const int u = unit_of(j);
      if (u >= 2 * T::UK) continue;  // whole waves
      // (Opaque, or the eight rows' sums are kept in registers of their own.)
      uint32_t at = uoff[j] + k0 * (u - lane < T::UK ? 1u : uint32_t(a.dim)) * 4u;
      asm("" : "+v"(at));
      if (u - lane < T::UK) {
#pragma unroll
        for (int e = 0; e < 8; ++e) raw[j][e] = ld4(krs, at + uint32_t(e) * uint32_t(a.cap) * 4u);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) raw[j][e] = ld4(vrs, at + (8u * (e >> 2) + (e & 3)) * uint32_t(a.dim) * 4u);
      }
    }
  };
  auto trim_tile = [&](int t) {
    const int k0 = t * KT;
    const bool inside = k0 >= klo && k0 + KT <= khi;  // uniform
    if (inside && a.dim == DP) return;
#pragma unroll
    for (int j = 0; j < T::NU; ++j) {
      const int u = unit_of(j);
      if (u >= 2 * T::UK) continue;
      if (u - lane < T::UK) {
        const int key = k0 + 4 * (u % (KT / 4));
        if (inside) continue;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float4 &v = raw[j][e];
          v.x = key >= klo && key < khi ? v.x : 0.0f;
          v.y = key + 1 >= klo && key + 1 < khi ? v.y : 0.0f;
          v.z = key + 2 >= klo && key + 2 < khi ? v.z : 0.0f;
          v.w = key + 3 >= klo && key + 3 < khi ? v.w : 0.0f;
        }
      } else {
        const int x = u - T::UK, ch = 4 * (x % (DP / 4)), kk = x / (DP / 4);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int key = k0 + 16 * (kk >> 1) + 8 * (e >> 2) + 4 * (kk & 1) + (e & 3);
          const int n = key >= klo && key < khi ? a.dim - ch : 0;  // channels from ch
          float4 &v = raw[j][e];
          v.x = n > 0 ? v.x : 0.0f;
          v.y = n > 1 ? v.y : 0.0f;
          v.z = n > 2 ? v.z : 0.0f;
          v.w = n > 3 ? v.w : 0.0f;
        }
      }
    }
  };
  // Largest magnitude bits of this wave's K units and V units.
  auto wave_max = [&](uint32_t &mk, uint32_t &mv) {
    mk = mv = 0;
#pragma unroll
    for (int j = 0; j < T::NU; ++j) {
      const int u = unit_of(j);
      if (u >= 2 * T::UK) continue;
      uint32_t m = 0;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        m = max(max(max(m, abs_bits(raw[j][e].x)), abs_bits(raw[j][e].y)),
                max(abs_bits(raw[j][e].z), abs_bits(raw[j][e].w)));
      if (u - lane < T::UK) mk = max(mk, m);
      else mv = max(mv, m);
    }
    mk = wave_umax(mk);
    mv = wave_umax(mv);
  };
  auto write_tile = [&](float ks, float vs) {
#pragma unroll
    for (int j = 0; j < T::NU; ++j) {
      const int u = unit_of(j);
      if (u >= 2 * T::UK) continue;
      const bool isk = u - lane < T::UK;
      const int x = isk ? u : u - T::UK;
      uint4 *dst;
      int plane;
      if (isk) {
        const int key = 4 * (x % (KT / 4)), o = x / (KT / 4);
        dst = kf + ((key >> 5) * T::DS + (o >> 1)) * 64 + (key & 31) + 32 * (o & 1);
        plane = T::KF;
      } else {
        const int ch = 4 * (x % (DP / 4)), kk = x / (DP / 4);
        dst = vf + ((ch >> 5) * T::KS + (kk >> 1)) * 64 + (ch & 31) + 32 * (kk & 1);
        plane = T::VF;
      }
      const float s = isk ? ks : vs;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
          v[e] = i == 0 ? raw[j][e].x : (i == 1 ? raw[j][e].y : (i == 2 ? raw[j][e].z : raw[j][e].w));
        planes8(v, s, dst[i], dst[plane + i]);
      }
    }
  };

  f32x16 acc[T::CB];
#pragma unroll
  for (int c = 0; c < T::CB; ++c)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[c][e] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;  // l_run: this half-wave's keys
  bool slow = false;
  int ev = -110;                          // exponent of V's planes, acc holds O 2^(kPExp - ev)

  if (tb < te) load_tile(tb);
  for (int t = tb; t < te; ++t) {
    const int par = t & 1;
    trim_tile(t);
    {
      uint32_t mk, mv;
      wave_max(mk, mv);
      if (lane == 0) {
        red[par][0][wave] = qbad ? kInfBits : mk;
        red[par][1][wave] = mv;
      }
    }
    __syncthreads();  // the maxima, and every wave is done with the previous tile's fragments
    uint32_t mk = max(max(red[par][0][0], red[par][0][1]), max(red[par][0][2], red[par][0][3]));
    uint32_t mv = max(max(red[par][1][0], red[par][1][1]), max(red[par][1][2], red[par][1][3]));
    if (mk >= kInfBits || mv >= kInfBits) {  // uniform: an infinity or NaN among the keys or in q
      slow = true;
      break;
    }
    const int ek = plane_exp(mk), ev_new = max(ev, plane_exp(mv));
    write_tile(ldexpf(1.0f, -ek), ldexpf(1.0f, -ev_new));
    if (t + 1 < te) load_tile(t + 1);
    __syncthreads();

    float s[T::KB][16];
    if (busy) {
      // ---- scores of this lane's row: keys 32 kb + 8 (i / 4) + 4 h + i % 4
      const float cf = ldexpf(qscale, ek);
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
          for (int i = 0; i < 16; ++i) s[kb][i] = d[i] * cf;
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
      float sum = 0.0f;
#pragma unroll
      for (int kb = 0; kb < T::KB; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[kb][i] = __expf(s[kb][i] - m_sub);
          sum += s[kb][i];
        }
      l_run = l_run * keep + sum;
      m_run = m_new;
      // acc to the new maximum and V's new exponent (skipped when no row changes)
      const float f = ldexpf(keep, max(ev - ev_new, -200));
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
        planes8(pv, 16384.0f, ph, pl);
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
    ev = ev_new;
  }
  if (slow) {
    // Infinities or NaNs among the keys would reach rows that do not see them
    // through the products' zeros, and in q would meet the zeros of the lower
    // planes (inf, which a soft cap makes finite, would be NaN): this part is
    // computed row by row instead, a wave per query row, in fp32 as k_attn does.
    for (int i = wave; i < kQRows && q0 + i < nq; i += 4) {
      const int row = (q0 + i) / a.group, hd = kh * a.group + (q0 + i) % a.group;
      const float *qr = a.q + (size_t(row) * a.heads + hd) * a.dim;
      const unsigned *mrow =
          reinterpret_cast<const unsigned *>(a.cache + 2 * size_t(a.cap) * width) + size_t(row) * a.cap;
      const float mul = a.scale > 0.0f ? a.scale : 1.0f / sqrtf(float(a.dim));
      float m = -INFINITY, l = 0.0f, o[2] = {0.0f, 0.0f};  // channels lane, lane + 64
      for (int key = max(first_key(row), tb * KT); key < min(a.position + row + 1, te * KT); ++key) {
        if (a.masked && mrow[key] == 0u) continue;
        float d = 0.0f;
        for (int c = lane; c < a.dim; c += 64) d += qr[c] * kt[size_t(c) * a.cap + key];
        float sc = dev::wave_sum_xor(d) * mul;
        if (a.softcap > 0.0f) sc = a.softcap * tanhf(fminf(fmaxf(sc / a.softcap, -20.0f), 20.0f));
        const float mn = fmaxf(m, sc);
        // (a NaN before any other key counts, too)
        const float kp = mn == -INFINITY ? 1.0f : expf(m - mn), w = sc == -INFINITY ? 0.0f : expf(sc - mn);
        l = l * kp + w;
        m = mn;
        for (int c = lane, j = 0; c < a.dim; c += 64, ++j) {
          const float add = w * vb[size_t(key) * a.dim + c];
          if (j == 0) o[0] = o[0] * kp + add;
          else o[1] = o[1] * kp + add;
        }
      }
      const size_t rh = size_t(row) * a.heads + hd;
      float *dst = a.splits == 1 ? a.out + rh * a.dim : a.opart + (size_t(split) * a.rows * a.heads + rh) * a.dim;
      for (int c = lane, j = 0; c < a.dim; c += 64, ++j) {
        const float v = j == 0 ? o[0] : o[1];
        dst[c] = a.splits == 1 ? v / l : v;
      }
      if (a.splits > 1 && lane == 0) {
        float *ml = a.ml + (size_t(split) * a.rows * a.heads + rh) * 2;
        ml[0] = m;
        ml[1] = l;
      }
    }
    return;
  }

  if (!qin || !busy) return;
  const float l = l_run + dev::xor_lanes<32>(l_run);
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
        v[e] = ldexpf(acc[c][4 * g + e], ev - kPExp);
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
      size_t(dim) * cap * 4 > 0x7FFFFFFFull ||  // 32-bit offsets within a KV head
      (long long)rows * heads * (window > 0 ? std::min(window, last_end) : last_end) < least)
    return false;
  p.qtiles = int((nq + kQRows - 1) / kQRows);
  // The keys of one workgroup's rows: at most the window and those rows.
  const int longest = window > 0 ? int(std::min<long long>((long long)window + kQRows, last_end)) : last_end;
  const int tiles = (longest + 63) / 64;
  // Two workgroups per CU (one where a tile is 64 keys of 96 channels, which
  // takes a SIMD's registers), at least two tiles of 64 keys each.
  const long long wgs = (long long)kv_heads * p.qtiles, target = std::max(1, tuning().attn_wgs) / (dim > 64 && dim <= 96 ? 2 : 1);
  p.splits = int(std::max<long long>(1, std::min<long long>(target / std::max<long long>(1, wgs), tiles / 2)));
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
  else if (dim <= 96) launch<96, 64>(a, s);
  else launch<128, 32>(a, s);
  hip_check(hipGetLastError(), "attention launch");
}

}  // namespace qnn
