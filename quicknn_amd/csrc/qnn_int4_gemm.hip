// qnn_int4_gemm.hip -- native INT4 projections of many rows (prompt chunks) on
// the fp16 matrix cores.
//
// The matvec kernels (qnn_int4.hip) take at most 16 rows per pass over the
// weight, so a 128-row call read, unpacked and combined every weight eight
// times.  Here a workgroup holds all rows of the call against 128 weight rows,
// and each packed weight is read from memory once.
//
//     C[m][n] = sum_g s[n][g] * sum_{k in group g} x[m][k] (q[n][k] - 8)
//
// * x is prepared once per call (k_i4_act): scaled per row by a power of two
//   and split into two fp16 values, hi = fp16(x'), lo = fp16((x' - hi) 2^11): 22
//   significant bits, against the 16 bits of the matvec's fixed point.
// * q - 8 is an exact fp16 integer, unpacked in registers: nibbles under the
//   exponent of 1024, then one packed fp16 add or fma (9 operations for 8
//   weights).
// * Per 32-element group and 32 x 32 tile, four v_mfma_f32_32x32x16_f16 (two
//   K-halves of hi, two of lo) give the group's sum from zero, and one fma per
//   output folds the group's fp32 scale, which is one register per lane
//   because a lane's results share a weight row.  The scales stay fp32 and no
//   weight is rounded.
// Measured against 64 bits the products are an order of magnitude closer than
// the matvec's (1e-7 of the result against 1e-5).
//
// What bounds it: no unit alone.  The matrix cores have 4 M N K operations (two
// fp16 planes; a SIMD of a full card retires one of these MFMAs in 18.5 ns, so a
// K-tile of 128 x 128 outputs takes 0.59 us at least and 0.85 us as built), and
// the ends of a workgroup (first loads, group halves, partial sums) take 4.4 us.
// Counters, gate/up pair at 128 rows: matrix cores busy 23 %, VALU (folds,
// unpacking) 32 % of the elapsed cycles, waves waiting 29 % of theirs; 38 MB read
// for 31 of weights, 30 MB of partial sums written.  Hence:
// * a workgroup is eight waves, two per SIMD, so that one's folds run under
//   the other's products: 2 (rows) x 2 (weight blocks of 64 rows) x 2 (the
//   two groups of a K-tile), the group halves meeting in LDS at the end;
// * everything arrives by loads that write LDS (no registers in flight), ST
//   K-tiles deep, as the activations come from L2 and the weights from HBM;
// * while a row block's MFMAs run (two independent chains), the wave reads the
//   next row block's fragments, folds the previous one's sums and unpacks the
//   next weights, a few operations after each MFMA (0.95 us per K-tile with
//   one chain, and literals in the unpacking).
// A K-range split over workgroups (few weight rows) leaves partial sums that
// k_i4_sum adds in slice order.  Results depend on the weight's shape only:
// not on the number of rows of the call, nor on whether gate and up run as
// one launch.
//
// Measured, 128 rows, weights rotated beyond the caches: gate/up pair of 2560
// -> 9728 39 us + 9 us of sums and 5 us of activations (the matvec kernels:
// 8 launches of 19 us), down 9728 -> 2560 21 + 6 + 8 us (8 x 12 us); a whole
// MLP layer with its norm and residual 259 -> 90 us, at 64 rows 135 -> 66, at
// 32 rows 73 -> 63 us.  K-slices of that pair: 1 51.5 us, 2 55.7, 3 49.2, 4
// 56.5, 5 54.6; of that down: 6 39.5, 8 36.3, 10 33.5, 12 34.2, 13 44.3 us.
// From how many rows (Tuning::i4_gemm_rows): an MLP layer at 17 rows takes
// 38.3 us here and 34.6 with the matvec kernels at 512 -> 1024 (59.9 and 58.5
// at 2560 -> 9728), at 24 rows 38.6 and 41.1 (61.4 and 61.0), at 32 rows 38.1
// and 46.9 (63.1 and 73.0): from 25.
#include <type_traits>

#include "qnn_int4_dev.h"

namespace qnn {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
using dev::half8;
using dev::I4Masks;
using dev::Rsrc;

// ---- activations ------------------------------------------------------------
// Piece (m32, g, plane, kk, lane) of 16 bytes: 8 halfs of row 32 m32 + lane %
// 32, group g, packed dword d = 2 (lane / 32) + kk of the group (elements 8d ..
// 8d+7) in the order 0 4 1 5 2 6 3 7 that unpacking a weight dword gives.
// Four rows per workgroup (so that a 64-byte segment of a piece is written at
// once), 256 threads each, and gridDim.y workgroups per four rows: every one
// reads its rows for their largest element, and writes its share of them (one
// workgroup per four rows leaves 32 for 128 rows: 13 us at 9728 elements).
// Rows past M, elements past K and the padding group (groups are padded to an
// even number) are zero.
__global__ __launch_bounds__(1024) void k_i4_act(const float *__restrict__ x, int M, int K, int stride, int gpad,
                                                 int *__restrict__ ex, uint4 *__restrict__ frag) {
  __shared__ float red[4][4];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, rw = wave >> 2, part = wave & 3;
  const int t = part * 64 + lane, row = blockIdx.x * 4 + rw;
  const bool in = row < M;
  const float *r = x + size_t(in ? row : 0) * stride;
  const bool vec = (stride & 3) == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
  const int chunks = 4 * gpad;
  auto load8 = [&](int c, float (&v)[8]) {
    const int k0 = 8 * c;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = 0.0f;
    if (!in) return;
    if (vec && k0 + 8 <= K) {
      const float4 a = *reinterpret_cast<const float4 *>(r + k0), b = *reinterpret_cast<const float4 *>(r + k0 + 4);
      v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (k0 + i < K) v[i] = r[k0 + i];
    }
  };
  float amax = 0.0f;
#pragma unroll 4
  for (int c = t; c < chunks; c += 256) {
    float v[8];
    load8(c, v);
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
  }
  const int c1 = chunks * (int(blockIdx.y) + 1) / int(gridDim.y), c0 = chunks * int(blockIdx.y) / int(gridDim.y) + t;
  float first[8];  // its share's first chunk travels with them
  if (c0 < c1) load8(c0, first);
  amax = dev::wave_max_xor(amax);
  if (lane == 0) red[rw][part] = amax;
  __syncthreads();
  const int e = dev::act_exp(fmaxf(fmaxf(red[rw][0], red[rw][1]), fmaxf(red[rw][2], red[rw][3])));
  if (t == 0 && blockIdx.y == 0) ex[row] = e;
  const float sc = ldexpf(1.0f, -e);
  auto put = [&](int c, const float (&v)[8]) {
    const int g = c >> 2, d = c & 3;
    uint4 *dst = frag + ((size_t(row >> 5) * gpad + g) * 4 + (d & 1)) * 64 + (row & 31) + 32 * (d >> 1);
    dev::act_planes(v, sc, dst[0], dst[128]);
  };
  if (c0 < c1) put(c0, first);
  for (int c = c0 + 256; c < c1; c += 256) {
    float v[8];
    load8(c, v);
    put(c, v);
  }
}

// ---- product ------------------------------------------------------------------
struct I4GemmArgs {
  I4Layout l;                 // one lane per row
  const uint8_t *w[2];        // the matrix; with a pair, gate and up
  const uint4 *frag;          // k_i4_act's pieces
  const int *ex;              // row exponents
  float *y, *g, *u;           // outputs [M][N] (g, u: a pair's two sums, y their GLU)
  float *part;                // K-split: partial sums [slice][matrix][M][N]
  int M, N, gpad, m32, tiles, slices, ktiles;
};

// 16 bytes per lane from global memory into LDS at `lds` (uniform).
// The compiler does not see the write: gemm_vmwait and the barriers order it.
// M0 is set before each load; nothing else here uses it.
__device__ __forceinline__ void gemm_dma16(Rsrc r, uint32_t lds, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(r),
               "s"(soff)
               : "memory");
}
template <int N>
__device__ __forceinline__ void gemm_vmwait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// A K-tile is two groups.  Stage: A [2 MB row blocks][2 groups][4] pieces of
// 1 KiB, the nibbles [2 blocks][2 groups] of 1 KiB, the scale pieces (four
// groups each) [2 blocks] of 1 KiB.
template <int MB>
struct I4Stage {
  static constexpr int AP = 16 * MB;        // A pieces
  static constexpr int APW = AP / 8;        // per wave
  static constexpr int LPW = APW + 1;       // loads per wave and K-tile
  static constexpr uint32_t B = AP * 1024, S = B + 4096, BYTES = S + 2048;
  static constexpr int ST = MB == 2 ? 4 : 6;  // stages: 152 KiB (128 rows), 132 KiB (64 rows)
};
constexpr uint32_t kI4EpiBytes = 64 * 1024;  // the epilogue's exchange: 8 waves x 32 floats per lane
template <int MB>
constexpr size_t i4_gemm_lds() {
  return size_t(I4Stage<MB>::BYTES) * I4Stage<MB>::ST;
}
static_assert(i4_gemm_lds<2>() <= 160 * 1024 && i4_gemm_lds<1>() >= kI4EpiBytes, "LDS of the INT4 GEMM");

// PAIR: weight block `unit` of the gate and of the up matrix; otherwise
// blocks 2 unit and 2 unit + 1 of one matrix.
template <int MB, bool PAIR>
__global__ __launch_bounds__(512) void k_i4_gemm(const I4GemmArgs a) {
  using SG = I4Stage<MB>;
  extern __shared__ uint4 lds[];
  // Slice-major order, an eighth of it per blockIdx % 8 (an XCD, as the device
  // usually deals them): an XCD's L2 then holds one or two K-slices of x.
  const int id = int(blockIdx.x & 7u) * int(gridDim.x >> 3) + int(blockIdx.x >> 3);
  if (id >= a.tiles * a.slices) return;
  const int slice = id / a.tiles, unit = id - slice * a.tiles;
  const int kt0 = slice * a.ktiles / a.slices, nkt = (slice + 1) * a.ktiles / a.slices - kt0;
  const int tid = threadIdx.x, lane = tid & 63, wave = dev::wave_id();
  const int wm = wave & 1, wn = (wave >> 1) & 1, kw = wave >> 2;
  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(lds));

  // ---- this wave's loads of a K-tile: APW pieces of A, and one nibble piece
  // (waves 0-3: block wave % 2, group wave / 2) or one scale piece (waves 4-7:
  // block wave % 2, two waves each).  The choice is in registers, not in a
  // branch, which would part the loop's products from its folds.
  const int lb = wave & 1, lg = (wave >> 1) & 1;
  const bool lscl = wave >= 4;
  const int lblk = PAIR ? unit : 2 * unit + lb;
  const bool lin = lblk < a.l.blocks;  // an odd number of blocks: the last one's partner reads nothing
  const uint32_t lbytes = uint32_t(lscl ? a.l.quads() : a.l.steps) * 1024u;  // per block
  const uint8_t *lbase = a.w[PAIR ? lb : 0] + (lscl ? a.l.nib_bytes() : 0) + size_t(lin ? lblk : 0) * lbytes;
  const uint32_t lsize = lin ? lbytes : 0u, lshift = lscl ? 2 : 0;
  const uint32_t ldst = lscl ? SG::S + uint32_t(lb) * 1024u : SG::B + uint32_t(lb * 2 + lg) * 1024u;
  const uint32_t abytes = uint32_t(a.m32) * uint32_t(a.gpad) * 4096u;
  // A piece wave * APW + i is (row block, group, i + its first of the 4).
  const int ap = wave * SG::APW;
  const uint32_t asoff = (uint32_t(ap >> 3) * uint32_t(a.gpad) + uint32_t((ap >> 2) & 1)) * 4096u + uint32_t(ap & 3) * 1024u;
  const uint32_t l16 = uint32_t(lane) * 16u;
  // Load i of K-tile kt of the slice into its stage; past the end every load
  // is out of its buffer's range (the count of outstanding loads stays the
  // same).
  auto load_one = [&](int kt, int i) {
    const bool live = kt < nkt;
    const uint32_t st = lds0 + uint32_t(kt % SG::ST) * SG::BYTES, ktg = uint32_t(kt0 + kt);
    if (i < SG::APW)
      gemm_dma16(dev::rsrc(a.frag, live ? abytes : 0u), __builtin_amdgcn_readfirstlane(st + uint32_t(ap + i) * 1024u),
                 l16, live ? asoff + ktg * 8192u + uint32_t(i) * 1024u : 0u);
    else
      gemm_dma16(dev::rsrc(lbase, live ? lsize : 0u), __builtin_amdgcn_readfirstlane(st + ldst), l16,
                 live ? ((2u * ktg + uint32_t(lg)) >> lshift) * 1024u : 0u);
  };
#pragma unroll
  for (int k = 0; k < SG::ST - 1; ++k)
#pragma unroll
    for (int i = 0; i < SG::LPW; ++i) load_one(k, i);

  const I4Masks masks = dev::i4_masks();
  float acc[MB][2][16];
  f32x16 d[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
#pragma unroll
      for (int i = 0; i < MB; ++i) acc[i][t][e] = 0.0f;
      d[0][t][e] = d[1][t][e] = 0.0f;
    }
  half8 af[MB][2][2];  // [row block][plane][kk]
  half8 bf[2][2][2][2];  // [K-tile parity][32-row half of the block][plane][kk]
  float sc[2][2] = {{0.0f, 0.0f}, {0.0f, 0.0f}};  // [K-tile parity][32-row half]

  auto stage_at = [&](int kt) { return reinterpret_cast<const uint8_t *>(lds) + uint32_t(kt % SG::ST) * SG::BYTES; };
  auto read_a = [&](half8 (&f)[2][2], const uint8_t *st, int i, int sub) {
    const uint4 v =
        *reinterpret_cast<const uint4 *>(st + uint32_t(((wm * MB + i) * 2 + kw) * 4 + sub) * 1024u + uint32_t(lane) * 16u);
    __builtin_memcpy(&f[sub >> 1][sub & 1], &v, 16);
  };
  auto read_raw = [&](const uint8_t *st) {
    return *reinterpret_cast<const uint4 *>(st + SG::B + uint32_t(wn * 2 + kw) * 1024u + uint32_t(lane) * 16u);
  };
  // The scales of this wave's group of K-tile kt (the slice's first K-tile may sit in the middle of a piece).
  auto read_s = [&](float (&f)[2], const uint8_t *st, int kt) {
    const float *s = reinterpret_cast<const float *>(st + SG::S + uint32_t(wn) * 1024u + uint32_t(lane & 31) * 16u) +
                     ((2 * (kt0 + kt) + kw) & 3);
    f[0] = s[0];
    f[1] = s[128];
  };
  // Row l's dwords (lane l) -> dword 2h + kk of row 32 t + lane % 32 (h = lane / 32).
  auto unpack_pair = [&](half8 (&f)[2][2][2], uint32_t d0, uint32_t d2, int kk) {
    const auto r = __builtin_amdgcn_permlane32_swap(d0, d2, false, false);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f[t][0][kk] = dev::unpack_i4(r[t], masks);
      f[t][1][kk] = dev::lower_i4(f[t][0][kk]);
    }
  };

  // One K-tile (P: its parity).  Phase i runs the 8 MFMAs of row block i, two
  // independent chains, and in their shadow folds the group sums of the phase
  // before, reads the row block of the phase after and (last phase) unpacks
  // the next K-tile's weights.
  auto tile = [&](auto P_, int kt) {
    constexpr int P = decltype(P_)::value, Q = P ^ 1;
    gemm_vmwait<SG::LPW *(SG::ST - 3)>();  // this wave's loads of K-tile kt + 1
    __syncthreads();                        // everybody's; and nobody reads K-tile kt - 1's stage any more
    const uint8_t *st0 = stage_at(kt), *st1 = stage_at(kt + 1);
    uint4 raw = make_uint4(0, 0, 0, 0);
    const f32x16 zero = {};
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      constexpr int LASTI = MB - 1;
      const int D = MB == 2 ? i : P;           // this phase's group sums
      const int pi = (i + MB - 1) % MB;        // the phase before's row block
      constexpr int S1 = MB == 2 ? P : Q;  // (of phases after the first) the phase before's K-tile parity
      if (i == LASTI) raw = read_raw(st1);
      half8 an[2][2];  // MB == 1: the next K-tile's row block
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int t = j & 1, p = j >> 2, kk = (j >> 1) & 1;
        d[D][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i][p][kk], bf[P][t][p][kk], j < 2 ? zero : d[D][t], 0, 0, 0);
        if (j < 4) {
          if (MB == 2) read_a(af[i ^ 1], i == 0 ? st0 : st1, i ^ 1, j);
          else read_a(an, st1, 0, j);
        }
        const int li = i * 8 + j;
        if (li % MB == 0 && li / MB < SG::LPW) load_one(kt + SG::ST - 1, li / MB);
        if (j >= 1) {
#pragma unroll
          for (int f = (j - 1) * 32 / 7; f < j * 32 / 7; ++f) {
            const int pt = f >> 4, e = f & 15;
            acc[pi][pt][e] = fmaf(d[D ^ 1][pt][e], sc[i == 0 ? Q : S1][pt], acc[pi][pt][e]);
            asm volatile("" : "+v"(acc[pi][pt][e]));  // here: sunk to the end, d would stay live past its next products
          }
        }
        if (i == LASTI && j == 4) unpack_pair(bf[Q], raw.x, raw.z, 0);
        if (i == LASTI && j == 6) unpack_pair(bf[Q], raw.y, raw.w, 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (i == LASTI) read_s(sc[Q], st1, kt + 1);  // its old values are folded
      if (MB == 1)
#pragma unroll
        for (int e = 0; e < 4; ++e) af[0][e >> 1][e & 1] = an[e >> 1][e & 1];
    }
  };

  gemm_vmwait<SG::LPW *(SG::ST - 2)>();
  __syncthreads();
  {
    const uint8_t *st = stage_at(0);
    const uint4 raw = read_raw(st);
    read_s(sc[0], st, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) read_a(af[0], st, 0, j);
    unpack_pair(bf[0], raw.x, raw.z, 0);
    unpack_pair(bf[0], raw.y, raw.w, 1);
  }
  int kt = 0;
  for (; kt + 1 < nkt; kt += 2) {
    tile(std::integral_constant<int, 0>(), kt);
    tile(std::integral_constant<int, 1>(), kt + 1);
  }
  auto fold_last = [&](const f32x16 (&ds)[2], const float (&ss)[2]) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[MB - 1][t][e] = fmaf(ds[t][e], ss[t], acc[MB - 1][t][e]);
  };
  if (kt < nkt) {
    tile(std::integral_constant<int, 0>(), kt);
    fold_last(MB == 1 ? d[0] : d[1], sc[0]);
  } else {
    fold_last(d[1], sc[1]);
  }

  // ---- the two group halves meet: wave kw keeps 32-row half t = kw of its
  // block and hands the other half over.
  gemm_vmwait<0>();  // no load writes LDS any more
  __syncthreads();
  float *xl = reinterpret_cast<float *>(lds);  // [wave][MB * 16][64]
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) xl[(wave * MB * 16 + i * 16 + e) * 64 + lane] = kw ? acc[i][0][e] : acc[i][1][e];
  __syncthreads();
  float v[MB][16];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float o = xl[((wave ^ 4) * MB * 16 + i * 16 + e) * 64 + lane];
      v[i][e] = kw ? o + acc[i][1][e] : acc[i][0][e] + o;  // group half 0 first
    }

  // Lane: weight row 32 kw + lane % 32 of block wn, x rows 8 (e / 4) + 4 (lane / 32) + e % 4.
  const int blk = PAIR ? unit : 2 * unit + wn, n = blk * 64 + 32 * kw + (lane & 31);
  auto row_of = [&](int i, int e) { return (wm * MB + i) * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3); };
  if (a.slices > 1) {
    if (n >= a.N) return;
    float *p = a.part + (size_t(slice) * (PAIR ? 2 : 1) + (PAIR ? wn : 0)) * a.M * a.N + n;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (row_of(i, e) < a.M) p[size_t(row_of(i, e)) * a.N] = v[i][e];
    return;
  }
  int ex[MB][16];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) ex[i][e] = a.ex[min(row_of(i, e), a.M - 1)];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) v[i][e] = ldexpf(v[i][e], ex[i][e]);
  if constexpr (PAIR) {
    __syncthreads();
    if (wn == 1)
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) xl[(wave * MB * 16 + i * 16 + e) * 64 + lane] = v[i][e];
    __syncthreads();
    if (n >= a.N) return;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = row_of(i, e);
        if (m >= a.M) continue;
        const size_t at = size_t(m) * a.N + n;
        if (wn == 1) {
          if (a.u != a.y) a.u[at] = v[i][e];  // a GLU written over the up sums: the GLU stays
        } else {
          a.g[at] = v[i][e];
          a.y[at] = dev::silu(v[i][e]) * xl[((wave | 2) * MB * 16 + i * 16 + e) * 64 + lane];
        }
      }
  } else {
    if (n >= a.N) return;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (row_of(i, e) < a.M) a.y[size_t(row_of(i, e)) * a.N + n] = v[i][e];
  }
}

// The K-slices' partial sums in slice order, scaled by the row's exponent;
// with a pair also the GLU.  V outputs of one row per thread.
template <bool PAIR, int V>
__global__ __launch_bounds__(256) void k_i4_sum(const I4GemmArgs a) {
  const size_t i = (size_t(blockIdx.x) * 256 + threadIdx.x) * V, count = size_t(a.M) * a.N;
  if (i >= count) return;
  const int e = a.ex[i / a.N];
  float s[PAIR ? 2 : 1][V];
#pragma unroll
  for (int m = 0; m < (PAIR ? 2 : 1); ++m)
#pragma unroll
    for (int j = 0; j < V; ++j) s[m][j] = 0.0f;
  for (int k = 0; k < a.slices; ++k)
#pragma unroll
    for (int m = 0; m < (PAIR ? 2 : 1); ++m) {
      const float *p = a.part + (size_t(k) * (PAIR ? 2 : 1) + m) * count + i;
      if constexpr (V == 4) {
        const float4 v = *reinterpret_cast<const float4 *>(p);
        s[m][0] += v.x, s[m][1] += v.y, s[m][2] += v.z, s[m][3] += v.w;
      } else {
        s[m][0] += p[0];
      }
    }
  auto put = [&](float *o, const float (&v)[V]) {
    if constexpr (V == 4) *reinterpret_cast<float4 *>(o + i) = make_float4(v[0], v[1], v[2], v[3]);
    else o[i] = v[0];
  };
#pragma unroll
  for (int m = 0; m < (PAIR ? 2 : 1); ++m)
#pragma unroll
    for (int j = 0; j < V; ++j) s[m][j] = ldexpf(s[m][j], e);
  if constexpr (PAIR) {
    float h[V];
#pragma unroll
    for (int j = 0; j < V; ++j) h[j] = dev::silu(s[0][j]) * s[1][j];
    put(a.g, s[0]);
    put(a.u, s[1]);
    put(a.y, h);
  } else {
    put(a.y, s[0]);
  }
}

int row_blocks(int rows) { return rows <= 64 ? 2 : 4; }  // 32-row blocks of the workgroup's tile

}  // namespace

I4GemmPlan int4_gemm_plan(const I4Layout &l, int rows) {
  I4GemmPlan p;
  p.gpad = (l.groups + 1) / 2 * 2;
  p.ktiles = p.gpad / 2;
  // K-slices: as many as give every CU a workgroup (a workgroup takes a CU's
  // LDS), at least 5 K-tiles each.  The count depends on the matrix alone,
  // so that a row's result does not depend on the call it is part of.
  const int tiles = (l.blocks + 1) / 2;
  p.slices = std::max(1, std::min(256 / std::max(1, tiles), p.ktiles / 5));
  p.frag_bytes = size_t(row_blocks(rows)) * p.gpad * 4096;
  p.part_bytes = p.slices > 1 ? size_t(p.slices) * rows * l.rows * 4 : 0;
  return p;
}

bool int4_gemm_applies(const I4Layout &l, int rows) {
  const Tuning &t = tuning();
  return t.i4_gemm_rows > 0 && rows >= t.i4_gemm_rows && rows <= 128 && t.i4_mfma != 0 && l.lanes == 1 &&
         l.groups <= kI4GemmMaxGroups && size_t(l.steps) * 1024 <= 0xFFFFFFFFull;
}

void int4_gemm_launch(const I4Launch &a, const I4GemmPlan &p, uint8_t *ws, hipStream_t s) {
  const bool pair = a.mode == I4_SWIGLU;
  if (pair && (!a.g_out || !a.u_out || !a.nib2)) fail(QNN_E_INVALID_OP, "int4 gemm pair without both matrices and sums");
  I4GemmArgs g;
  g.l = a.l;
  g.w[0] = static_cast<const uint8_t *>(a.nib);
  g.w[1] = static_cast<const uint8_t *>(a.nib2);
  int *ex = reinterpret_cast<int *>(ws);
  uint4 *frag = reinterpret_cast<uint4 *>(ws + kI4GemmExpBytes);
  g.ex = ex;
  g.frag = frag;
  g.part = reinterpret_cast<float *>(ws + kI4GemmExpBytes + p.frag_bytes);
  g.y = a.y;
  g.g = a.g_out;
  g.u = a.u_out;
  g.M = a.m;
  g.N = a.n;
  g.gpad = p.gpad;
  g.m32 = row_blocks(a.m);
  g.tiles = pair ? a.l.blocks : (a.l.blocks + 1) / 2;
  g.slices = p.slices;
  g.ktiles = p.ktiles;
  hipLaunchKernelGGL(k_i4_act, dim3(g.m32 * 8, (p.gpad + 63) / 64), dim3(1024), 0, s, a.x, a.m, a.k, a.x_stride, p.gpad, ex, frag);
  static const hipError_t attr = [] {
    const std::pair<const void *, size_t> k[] = {
        {reinterpret_cast<const void *>(&k_i4_gemm<1, false>), i4_gemm_lds<1>()},
        {reinterpret_cast<const void *>(&k_i4_gemm<1, true>), i4_gemm_lds<1>()},
        {reinterpret_cast<const void *>(&k_i4_gemm<2, false>), i4_gemm_lds<2>()},
        {reinterpret_cast<const void *>(&k_i4_gemm<2, true>), i4_gemm_lds<2>()}};
    for (const auto &f : k) {
      const hipError_t e = hipFuncSetAttribute(f.first, hipFuncAttributeMaxDynamicSharedMemorySize, int(f.second));
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }();
  hip_check(attr, "int4 gemm LDS size");
  const dim3 grid((size_t(g.tiles) * g.slices + 7) / 8 * 8), block(512);
  if (g.m32 == 2) {
    if (pair) hipLaunchKernelGGL((k_i4_gemm<1, true>), grid, block, i4_gemm_lds<1>(), s, g);
    else hipLaunchKernelGGL((k_i4_gemm<1, false>), grid, block, i4_gemm_lds<1>(), s, g);
  } else {
    if (pair) hipLaunchKernelGGL((k_i4_gemm<2, true>), grid, block, i4_gemm_lds<2>(), s, g);
    else hipLaunchKernelGGL((k_i4_gemm<2, false>), grid, block, i4_gemm_lds<2>(), s, g);
  }
  if (g.slices > 1) {
    const size_t count = size_t(g.M) * g.N;
    auto aligned = [](const float *q) { return reinterpret_cast<uintptr_t>(q) % 16 == 0; };
    const bool vec = g.N % 4 == 0 && aligned(g.y) && (!pair || (aligned(g.g) && aligned(g.u)));
    const dim3 sgrid((count / (vec ? 4 : 1) + 255) / 256);
    if (pair) {
      if (vec) hipLaunchKernelGGL((k_i4_sum<true, 4>), sgrid, dim3(256), 0, s, g);
      else hipLaunchKernelGGL((k_i4_sum<true, 1>), sgrid, dim3(256), 0, s, g);
    } else {
      if (vec) hipLaunchKernelGGL((k_i4_sum<false, 4>), sgrid, dim3(256), 0, s, g);
      else hipLaunchKernelGGL((k_i4_sum<false, 1>), sgrid, dim3(256), 0, s, g);
    }
  }
  hip_check(hipGetLastError(), "int4 gemm launch");
}

}  // namespace qnn
