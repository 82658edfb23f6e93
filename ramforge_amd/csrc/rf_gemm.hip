// rf_gemm.hip — the prefill GEMM for chunks of more than a few token tiles:
// Y[t][r] = sum_k W[r][k] X[t][k] on the packed layout of Q8_0 / Q4_0 / Q4_K /
// Q6_K (rf_matvec_packed.hip), split-K partials for rf_prefill.hip's reduces.
//
// The arithmetic is mm_packed's (rf_prefill.hip): exact integer codes in bf16
// times x in three bf16 pieces on the matrix cores, the block scale applied in
// f32 to each block's partial sum.  What differs is who does what how often:
//   * x is split once per launch (mm_split_x) into planes laid out as the
//     MFMA's A operand reads them: [32-element block][half][token tile][piece]
//     [lane][8], one contiguous KiB per wavefront load, straight to registers.
//     The pieces are truncations (8 significant bits each), so hi + mid + lo is
//     x exactly.
//   * a workgroup of four wavefronts decodes 256 weight rows of a 64-element
//     stage into LDS once, as bf16 in B operand order, for all its tokens
//     (WM wavefronts of 32 tokens).
//   * a 32 x 32 tile takes 192 matrix cycles for a block of 32 elements and 16
//     scale FMAs (64 VALU cycles).  Q8_0 and Q4_0 use v_mfma_f32_16x16x32_bf16:
//     two short chains per 16-row tile leave the registers for a pipeline in
//     which the scale FMAs, the LDS reads and the decode run under the MFMAs
//     (stage_k32), where the compiler runs the chain, its FMAs and the next LDS
//     read in turn (28672 x 4096, 512 tokens: matrix cores busy 51% of the
//     cycles for Q8_0, 53% for Q4_0; 39% for Q6_K, left to the compiler).  Q8_0
//     on one chip, 32 x 32 x 16 against this: 28672 x 4096, 512 tokens 381 and
//     353 us, 128 tokens 117 and 105; 6144 x 4096, 96 tokens 44.0 and 39.4;
//     4096 x 14336, 512 tokens 197 and 182.
//   * Q4_K and Q6_K stay with v_mfma_f32_32x32x16_bf16: Q6_K has a scale per 16
//     elements, half a 16 x 16 x 32 operand, and Q4_K's mins want the
//     32 x 32 x 2 f32 form (as 16 x 16 x 4 the matrix time of two stages' mins
//     is the same and the registers spill: 28672 x 4096, 512 tokens 390 us
//     either way, 4096 x 14336, 96 tokens 67 and 72).
//   * the x planes and the scales of odd 32-element blocks carry a minus sign:
//     the matrix cores' chained sums round towards minus infinity, which would
//     add up over a row (a mean error of 0.7 of the rms one at K = 14336; with the
//     signs 0.03) and so takes itself off.
// A wavefront owns 32 tokens x TN row tiles: the x planes (the larger operand,
// three pieces) are read by one wavefront only, the weights by all from LDS.
#include "rf_gemm.h"
#include "rf_kernels.h"

namespace rf {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t GT_ROWS = 256, GT_THREADS = 256;
constexpr uint32_t GT_FRAG = 64 * 16;            // bytes of one operand fragment (32 rows x 16 elements of bf16)
constexpr uint32_t GT_B = GT_ROWS / 32 * 4 * GT_FRAG;  // bytes of one stage of decoded weights
constexpr uint32_t GT_OOR = 0xFFFFFFF0u;
constexpr int GT_RSRC_WORD3 = 0x00020000;
typedef __amdgpu_buffer_rsrc_t GtRsrc;

__device__ __forceinline__ uint4 gt_ld16(GtRsrc r, uint32_t off) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
  return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ uint32_t gt_ld4(GtRsrc r, uint32_t off) {
  return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
}
__device__ __forceinline__ uint32_t gt_ld2(GtRsrc r, uint32_t off) {
  return (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0);
}

// Four signed bytes as two words of bf16 pairs: every code is exact in the
// upper half of its float.
__device__ __forceinline__ uint2 gt_bf16(uint32_t w) {
  const uint32_t a = __float_as_uint(rf_sb(w, 0)), b = __float_as_uint(rf_sb(w, 1));
  const uint32_t c = __float_as_uint(rf_sb(w, 2)), d = __float_as_uint(rf_sb(w, 3));
  return make_uint2(__builtin_amdgcn_perm(b, a, 0x07060302u), __builtin_amdgcn_perm(d, c, 0x07060302u));
}

// LDS byte of piece (row, 16-element quarter kq, 8-element half h) of a stage.
// K32 (operands of 16 rows x 32 elements): fragment (row / 16, kq / 2), slot
// 16 (2 (kq % 2) + h) + row % 16; otherwise (32 rows x 16 elements) fragment
// (row / 32, kq), slot 32 h + row % 32.  The slot's low bits are permuted by
// kq, so that the lanes of a store (two or four rows x the quarters a lane
// holds) and of a fragment read (64 consecutive slots) hit distinct banks.
__device__ __forceinline__ uint32_t gt_swz(uint32_t kq) { return (0x2640u >> (4u * kq)) & 0xFu; }
template <bool K32>
__device__ __forceinline__ uint32_t gt_slot(uint32_t row, uint32_t kq, uint32_t h) {
  if constexpr (K32)
    return ((row >> 4) * 2u + (kq >> 1)) * GT_FRAG + ((32u * (kq & 1u) + 16u * h + (row & 15u)) ^ gt_swz(kq)) * 16u;
  else
    return ((row >> 5) * 4u + kq) * GT_FRAG + ((32u * h + (row & 31u)) ^ gt_swz(kq)) * 16u;
}
// 8 codes (two words of bytes) of (row, kq, h)
template <bool K32>
__device__ __forceinline__ void gt_put8(uint8_t* b, uint32_t row, uint32_t kq, uint32_t h, uint32_t w0, uint32_t w1) {
  const uint2 lo = gt_bf16(w0), hi = gt_bf16(w1);
  *reinterpret_cast<uint4*>(b + gt_slot<K32>(row, kq, h)) = make_uint4(lo.x, lo.y, hi.x, hi.y);
}
// 16 codes (four words of bytes) of (row, kq), 32 x 16 fragments
__device__ __forceinline__ void gt_put16(uint8_t* b, uint32_t row, uint32_t kq, const uint32_t (&w)[4]) {
#pragma unroll
  for (uint32_t h = 0; h < 2; ++h) gt_put8<false>(b, row, kq, h, w[2 * h], w[2 * h + 1]);
}
__device__ __forceinline__ uint32_t gt_word(const uint4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// One stage (64 elements of 256 rows) of a format: load() requests a thread's
// share of the codes and row tid's scales into registers, put() decodes them
// into LDS: codes as bf16, NS scales per row (one per block of 32 elements,
// the second block's negated; Q6_K one per 16), Q4_K also its two mins.  K32
// formats store one of a thread's eight 16-byte pieces at a time and its row's
// scales apart.  Rows past the segment read as zeros.
template <uint32_t T> struct GtW;

// the low or high nibbles q of a word's bytes as signed bytes 16 (q - 8): the
// scale takes the 16 off
__device__ __forceinline__ uint32_t gt_top_nibbles(uint32_t w, int hi) {
  return rf_opaque(hi ? (w & 0xF0F0F0F0u) ^ 0x80808080u : rf_top_signed(w, 4));
}

template <> struct GtW<T_Q8_0> {
  static constexpr int NREG = 2, NS = 2;
  static constexpr bool MIN = false, K32 = true;
  uint4 c[4];
  uint32_t sc[2];
  __device__ __forceinline__ void load(const GtRsrc* rs, uint32_t row0, uint32_t rows, uint32_t s, uint32_t K,
                                       uint32_t tid) {
    const uint32_t nb = K / 32u;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
      const uint32_t r = row0 + i * 64u + (tid >> 2);
      c[i] = gt_ld16(rs[0], r < rows ? r * K + s * 64u + 16u * (tid & 3u) : GT_OOR);
    }
    const uint32_t r = row0 + tid;
#pragma unroll
    for (uint32_t b = 0; b < 2; ++b) sc[b] = gt_ld2(rs[1], r < rows && 2u * s + b < nb ? (r * nb + 2u * s + b) * 2u : GT_OOR);
  }
  __device__ __forceinline__ void put(int j, uint8_t* b, uint32_t tid) const {
    const int i = j >> 1, h = j & 1;
    gt_put8<true>(b, i * 64u + (tid >> 2), tid & 3u, h, gt_word(c[i], 2 * h), gt_word(c[i], 2 * h + 1));
  }
  __device__ __forceinline__ void scales(float* ds, uint32_t tid) const {
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) ds[k * GT_ROWS + tid] = (k ? -1.f : 1.f) * rf_half_to_float_fast(sc[k]);
  }
};

template <> struct GtW<T_Q4_0> {
  static constexpr int NREG = 2, NS = 2;
  static constexpr bool MIN = false, K32 = true;
  uint4 c[2];
  uint32_t sc[2];
  __device__ __forceinline__ void load(const GtRsrc* rs, uint32_t row0, uint32_t rows, uint32_t s, uint32_t K,
                                       uint32_t tid) {
    const uint32_t nb = K / 32u;
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
      const uint32_t r = row0 + i * 128u + (tid >> 1);
      c[i] = gt_ld16(rs[0], r < rows ? (r * nb + 2u * s + (tid & 1u)) * 16u : GT_OOR);
    }
    const uint32_t r = row0 + tid;
#pragma unroll
    for (uint32_t b = 0; b < 2; ++b) sc[b] = gt_ld2(rs[1], r < rows && 2u * s + b < nb ? (r * nb + 2u * s + b) * 2u : GT_OOR);
  }
  __device__ __forceinline__ void put(int j, uint8_t* b, uint32_t tid) const {
    const int i = j >> 2, hi = (j >> 1) & 1, h = j & 1;
    gt_put8<true>(b, i * 128u + (tid >> 1), 2u * (tid & 1u) + hi, h, gt_top_nibbles(gt_word(c[i], 2 * h), hi),
                  gt_top_nibbles(gt_word(c[i], 2 * h + 1), hi));
  }
  __device__ __forceinline__ void scales(float* ds, uint32_t tid) const {
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) ds[k * GT_ROWS + tid] = rf_half_to_float_fast(sc[k]) * (k ? -0.0625f : 0.0625f);
  }
};

// A stage is two sub-blocks: 32 bytes of qs, the low nibbles the first.  The
// codes are centred: d q - m = d (q - 8) + (8 d - m), so the sums of q - 8
// and of x that meet in the accumulator are small together.
template <> struct GtW<T_Q4_K> {
  static constexpr int NREG = 2, NS = 2;
  static constexpr bool MIN = true, K32 = false;
  uint4 c[2];
  uint4 h;  // row tid's header: d | dmin << 16, scale bytes 0-3, 4-7, 8-11
  __device__ __forceinline__ void load(const GtRsrc* rs, uint32_t row0, uint32_t rows, uint32_t s, uint32_t K,
                                       uint32_t tid) {
    const uint32_t nb = K / 256u;
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
      const uint32_t r = row0 + i * 128u + (tid >> 1);
      c[i] = gt_ld16(rs[0], r < rows ? (r * nb + (s >> 2)) * 128u + 32u * (s & 3u) + 16u * (tid & 1u) : GT_OOR);
    }
    const uint32_t r = row0 + tid;
    h = gt_ld16(rs[1], r < rows ? (r * nb + (s >> 2)) * 16u : GT_OOR);
  }
  __device__ __forceinline__ void put(uint8_t* b, float* ds, float* ms, uint32_t s, uint32_t tid) const {
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
      const uint32_t w[4] = {c[i].x, c[i].y, c[i].z, c[i].w};
      uint32_t lo[4], hi[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        lo[k] = rf_opaque(rf_top_signed(w[k], 4));
        hi[k] = rf_opaque((w[k] & 0xF0F0F0F0u) ^ 0x80808080u);
      }
      const uint32_t row = i * 128u + (tid >> 1), q = tid & 1u;
      gt_put16(b, row, q, lo);
      gt_put16(b, row, 2u + q, hi);
    }
    // get_scale_min (quant.rs:216-226) of sub-blocks 2 (s % 4), + 1
    const float d = rf_half_to_float_fast(h.x & 0xFFFFu), dmin = rf_half_to_float_fast(h.x >> 16);
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) {
      const uint32_t sh = 8u * (2u * (s & 1u) + k);  // byte (j & 3) of the 4-byte groups, j = 2 (s % 4) + k
      const uint32_t y = h.y >> sh, z = h.z >> sh, w = h.w >> sh;
      const bool low = (s & 3u) < 2u;  // uniform
      const uint32_t sc = low ? y & 63u : (w & 0xFu) | ((y >> 6) & 3u) << 4;
      const uint32_t mn = low ? z & 63u : ((w >> 4) & 0xFu) | ((z >> 6) & 3u) << 4;
      const float d1 = d * (float)sc;
      ds[k * GT_ROWS + tid] = d1 * (k ? -0.0625f : 0.0625f);
      ms[k * GT_ROWS + tid] = 8.f * d1 - dmin * (float)mn;
    }
  }
};

// A stage is two quarters (2 p, 2 p + 1) of a 128-element half: elements
// l = 0..31 of both, low bits in nibble p of ql bytes l and 32 + l, bits
// 2 (2 p + i) of qh byte l.
template <> struct GtW<T_Q6_K> {
  static constexpr int NREG = 4, NS = 4;
  static constexpr bool MIN = false, K32 = false;
  uint4 ql[2][2], qh[2];
  uint32_t sc, d;
  __device__ __forceinline__ void load(const GtRsrc* rs, uint32_t row0, uint32_t rows, uint32_t s, uint32_t K,
                                       uint32_t tid) {
    const uint32_t nb = K / 256u, hh = (s >> 1) & 1u;
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
      const uint32_t r = row0 + i * 128u + (tid >> 1), blk = r * nb + (s >> 2), j = 16u * (tid & 1u);
      const bool ok = r < rows;
      ql[i][0] = gt_ld16(rs[0], ok ? blk * 128u + 64u * hh + j : GT_OOR);
      ql[i][1] = gt_ld16(rs[0], ok ? blk * 128u + 64u * hh + 32u + j : GT_OOR);
      qh[i] = gt_ld16(rs[1], ok ? blk * 64u + 32u * hh + j : GT_OOR);
    }
    const uint32_t r = row0 + tid, blk = r * nb + (s >> 2);
    sc = gt_ld4(rs[2], r < rows ? blk * 16u + 4u * (s & 3u) : GT_OOR);
    d = gt_ld2(rs[3], r < rows ? blk * 2u : GT_OOR);
  }
  // 4 (q - 32) as a signed byte, the scale takes the 4 off
  __device__ __forceinline__ void put(uint8_t* b, float* ds, float*, uint32_t s, uint32_t tid) const {
    const uint32_t p = s & 1u;
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
      const uint32_t hq[4] = {qh[i].x, qh[i].y, qh[i].z, qh[i].w};
#pragma unroll
      for (uint32_t k = 0; k < 2; ++k) {
        const uint4 lv = ql[i][k];
        const uint32_t l[4] = {lv.x, lv.y, lv.z, lv.w};
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t low = (l[e] >> (4u * p)) & 0x0F0F0F0Fu, high = (hq[e] >> (4u * p + 2u * k)) & 0x03030303u;
          w[e] = rf_opaque(((low << 2) | (high << 6)) ^ 0x80808080u);
        }
        gt_put16(b, i * 128u + (tid >> 1), 2u * k + (tid & 1u), w);
      }
    }
    const float dd = rf_half_to_float_fast(d) * 0.25f;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) ds[k * GT_ROWS + tid] = (k < 2 ? dd : -dd) * rf_sb(sc, (int)k);
  }
};

struct GtSeg {
  const uint8_t* reg[PK_MAX_REGIONS];
  uint64_t bytes[PK_MAX_REGIONS];
  uint32_t rows, group_begin, col;
};
struct GtArgs {
  GtSeg seg[3];
  uint32_t nseg, n, ntt, K, nstages, spp, mtot, mtiles, groups, nsplit;
  const __bf16* planes;  // [2 nstages][2][ntt][3][64][8]
  const float* sums;     // [2 nstages][32 ntt] (Q4_K)
  float* part;           // [nsplit][n][mtot]
};

template <uint32_t T, int WM>
__global__ __launch_bounds__(GT_THREADS, 2) void mm_tile(GtArgs a) {
  typedef GtW<T> W;
  constexpr int TN = 2 * WM;       // 32-row tiles of a wavefront: 4 / WM wavefronts share 256 rows
  constexpr int RT = 2 * TN;       // the same in 16-row tiles
  constexpr bool K32 = W::K32;     // 16 x 16 x 32 operands, else 32 x 32 x 16
  __shared__ __align__(16) uint8_t bs[2][GT_B];
  __shared__ float ds[2][W::NS * GT_ROWS];
  __shared__ float ms[2][W::MIN ? 2 * GT_ROWS : 1];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t l32 = lane & 31u, lh = lane >> 5;
  const uint32_t wm = wave % WM, wn = wave / WM;
  // Workgroups go to the eight XCDs in turn: each XCD takes a run of
  // consecutive items, token tiles of one row group first, so that the tiles
  // that read the same weights share an L2.
  const uint32_t per = (gridDim.x + 7u) / 8u, big = gridDim.x - 8u * (per - 1u);  // XCDs 0 .. big - 1 take per items
  const uint32_t xcd = blockIdx.x & 7u, idx = blockIdx.x >> 3;
  const uint32_t item = xcd < big ? xcd * per + idx : big * per + (xcd - big) * (per - 1u) + idx;
  const uint32_t mt = item % a.mtiles, rest = item / a.mtiles, grp = rest % a.groups, sp = rest / a.groups;
  GtSeg s = a.seg[0];
  if (a.nseg > 1 && grp >= a.seg[1].group_begin) s = a.seg[1];
  if (a.nseg > 2 && grp >= a.seg[2].group_begin) s = a.seg[2];
  const uint32_t row0 = (grp - s.group_begin) * GT_ROWS, K = a.K;
  const uint32_t s0 = sp * a.spp, s1 = min(a.nstages, s0 + a.spp);
  GtRsrc rs[W::NREG];
#pragma unroll
  for (int k = 0; k < W::NREG; ++k)
    rs[k] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(s.reg[k]), 0, (int32_t)s.bytes[k], GT_RSRC_WORD3);
  const uint32_t tt = min(mt * WM + wm, a.ntt - 1u);  // a tile past the tokens computes the last one again
  const bf16x8* ap = reinterpret_cast<const bf16x8*>(a.planes) + (size_t)tt * 192u;
  const size_t kstride = (size_t)a.ntt * 192u;  // 16-byte pieces per 16 elements of k
  auto load_a = [&](bf16x8 (&v)[2][3], uint32_t blk) {
#pragma unroll
    for (uint32_t h = 0; h < 2; ++h)
#pragma unroll
      for (uint32_t p = 0; p < 3; ++p) v[h][p] = (ap + (2u * blk + h) * kstride + p * 64u)[lane];
  };

  // K32: acc[i][8 r + 4 f + e] is 16-row tile 2 i + r, token 16 f + 4 (lane / 16)
  // + e, row lane % 16; else 32-row tile i, token 8 (e / 4) + 4 lh + e % 4, row l32
  f32x16 acc[TN];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
  const f32x16 zero = acc[0];

  // One stage of K32 formats, from buffer buf: 2 RT groups, (block, 16-row
  // tile) in turn, of six MFMAs each (two token tiles x three pieces, smallest
  // first).  Written as a pipeline, as the compiler would run each chain, its
  // scale FMAs and the next LDS read one after the other: group g's MFMAs are
  // interleaved with group g - 1's scale FMAs and a share of the next stage's
  // decode, its operands were requested two groups before.
  const uint32_t l16 = lane & 15u;
  const uint32_t slot0 = (lane ^ gt_swz(lane >> 5)) * 16u, slot1 = (lane ^ gt_swz(2u + (lane >> 5))) * 16u;
  auto stage_k32 = [&](uint32_t buf, bf16x8 (&a0)[2][3], bf16x8 (&a1)[2][3], uint32_t next_a, auto&& decode) {
    bf16x8 b[3];
    float d[4];
    f32x4 t[2][2];
    const uint8_t* bb = &bs[buf][wn * RT * 2u * GT_FRAG];
    const float* db = &ds[buf][wn * RT * 16u + l16];
    auto fetch = [&](int g) {
      const int blk = g / RT, rt = g % RT;
      b[g % 3] = *reinterpret_cast<const bf16x8*>(bb + (blk ? slot1 : slot0) + (rt * 2 + blk) * GT_FRAG);
      d[g % 4] = db[blk * GT_ROWS + rt * 16];
    };
    auto mfma = [&](int g, int k) {  // k-th of the group: piece 2 - k / 2 of token tile k % 2
      const int f = k & 1, p = 2 - (k >> 1);
      f32x4& c = t[g & 1][f];
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g < RT ? a0[f][p] : a1[f][p], b[g % 3],
                                                  k < 2 ? f32x4{0.f, 0.f, 0.f, 0.f} : c, 0, 0, 0);
    };
    auto scale = [&](int g, int f, int e) {
      f32x16& c = acc[g % RT / 2];
      const int k = 8 * (g & 1) + 4 * f + e;
      c[k] = fmaf(d[g % 4], t[g & 1][f][e], c[k]);
    };
    fetch(0);
    fetch(1);
#pragma unroll
    for (int g = 0; g < 2 * RT; ++g) {
      if (g + 2 < 2 * RT) fetch(g + 2);
      mfma(g, 0);
      mfma(g, 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (g > 0) {
          scale(g - 1, k >> 1, 2 * (k & 1));
          scale(g - 1, k >> 1, 2 * (k & 1) + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        mfma(g, 2 + k);
      }
      if (g == RT - 1) load_a(a0, next_a);
      if (g >= RT) decode(g - RT);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) scale(2 * RT - 1, k >> 2, k & 3);
  };
  // block `blk` of the stage in buffer buf, 32 x 32 x 16 operands
  auto block_k16 = [&](uint32_t buf, uint32_t blk, const bf16x8 (&v)[2][3]) {
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const uint32_t rt = wn * TN + i;
      bf16x8 b[2];
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h) {
        const uint32_t kq = 2u * blk + h;
        b[h] = *reinterpret_cast<const bf16x8*>(&bs[buf][(rt * 4u + kq) * GT_FRAG + (lane ^ gt_swz(kq)) * 16u]);
      }
      if constexpr (W::NS == 4) {  // a scale per 16 elements
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
          f32x16 t = zero;
#pragma unroll
          for (int p = 2; p >= 0; --p) t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v[h][p], b[h], t, 0, 0, 0);
          const float d = ds[buf][(2u * blk + h) * GT_ROWS + rt * 32u + l32];
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][e] = fmaf(d, t[e], acc[i][e]);
        }
      } else {
        f32x16 t = zero;
#pragma unroll
        for (int p = 2; p >= 0; --p)  // the smallest pieces first
#pragma unroll
          for (uint32_t h = 0; h < 2; ++h) t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v[h][p], b[h], t, 0, 0, 0);
        const float d = ds[buf][blk * GT_ROWS + rt * 32u + l32];
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = fmaf(d, t[e], acc[i][e]);
      }
    }
  };

  // The partials are added up in `part` every `chain` stages: chains of at most 48
  // scale FMAs round no worse than mm_packed's split sums (relative error
  // against 64 bits at 28672 x 4096, 512 tokens: 1.3e-7; one chain of 128
  // 2.2e-7, mm_packed 1.4e-7) and cost 3% of the launch.
  const uint32_t tb = (mt * WM + wm) * 32u;
  const GtRsrc pr = __builtin_amdgcn_make_buffer_rsrc(
      a.part + ((size_t)sp * a.n + min(tb, a.n)) * a.mtot + s.col, 0,
      tb < a.n ? (int32_t)(((min(a.n - tb, 32u) - 1u) * a.mtot + s.rows) * 4u) : 0, GT_RSRC_WORD3);
  auto flush = [&](bool first) {
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      // offsets past the tokens or the segment's rows write nothing; opaque,
      // so that they are computed here and not kept through the stages
      const uint32_t r = row0 + (wn * TN + i) * 32u + (K32 ? l16 : l32), ld = rf_opaque(a.mtot * 4u);
      const uint32_t o0 = r < s.rows ? 4u * (K32 ? lane >> 4 : lh) * ld + r * 4u : GT_OOR;
      auto off = [&](int e) -> uint32_t {
        if constexpr (K32)
          return r + 16u * (e >> 3) < s.rows ? o0 + (16u * ((e >> 2) & 1) + (e & 3)) * ld + 64u * (e >> 3) : GT_OOR;
        else
          return r < s.rows ? o0 + (8u * (e / 4) + e % 4) * ld : GT_OOR;
      };
      if (!first) {  // uniform
        float old[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) old[e] = __uint_as_float(gt_ld4(pr, off(e)));
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] += old[e];
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[i][e]), pr, off(e), 0, 0);
        acc[i][e] = 0.f;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  constexpr uint32_t CHAIN = 48 / W::NS;
  const uint32_t parts = (s1 - s0 + CHAIN - 1u) / CHAIN, chain = (s1 - s0 + parts - 1u) / parts;

  W w;
  bf16x8 a0[2][3], a1[2][3];
  auto put_all = [&](uint32_t buf, uint32_t st) {  // the stage in w
    if constexpr (K32) {
#pragma unroll
      for (int j = 0; j < 8; ++j) w.put(j, bs[buf], tid);
      w.scales(ds[buf], tid);
    } else {
      w.put(bs[buf], ds[buf], ms[buf], st, tid);
    }
  };
  w.load(rs, row0, s.rows, s0, K, tid);
  load_a(a0, 2u * s0);
  put_all(0, s0);
  __syncthreads();
  for (uint32_t c0 = s0; c0 < s1; c0 += chain) {
    const uint32_t c1 = min(s1, c0 + chain);
    for (uint32_t st = c0; st < c1; ++st) {
      const uint32_t buf = (st - s0) & 1u, nx = min(st + 1u, s1 - 1u);  // the last stage requests itself again
      w.load(rs, row0, s.rows, nx, K, tid);
      load_a(a1, 2u * st + 1u);
      // the next stage's buffer: its last readers passed the barrier before
      if constexpr (K32) {
        stage_k32(buf, a0, a1, 2u * nx, [&](int r) {
#pragma unroll
          for (int j = r * 9 / RT; j < (r + 1) * 9 / RT; ++j) {
            if (j < 8) w.put(j, bs[buf ^ 1u], tid);
            else w.scales(ds[buf ^ 1u], tid);
          }
        });
      } else {
        float sx = 0.f;
        if constexpr (W::MIN) sx = a.sums[(size_t)(2u * st + lh) * a.ntt * 32u + tt * 32u + l32];
        block_k16(buf, 0, a0);
        load_a(a0, 2u * nx);
        block_k16(buf, 1, a1);
        if constexpr (W::MIN) {  // plus 8 d - m times the block's sum of x: f32 products on the matrix cores
#pragma unroll
          for (int i = 0; i < TN; ++i)
            acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(sx, ms[buf][lh * GT_ROWS + (wn * TN + i) * 32u + l32], acc[i], 0, 0, 0);
        }
        put_all(buf ^ 1u, nx);
      }
      __syncthreads();
    }
    flush(c0 == s0);
  }
}

// x [n][ldx] into the planes of mm_tile: one wavefront per (token tile,
// 32-element block), odd blocks negated; tokens past n and elements past K are
// zeros.  K32: fragment h is 16 tokens x 32 elements, else 32 x 16.  SUMS (not
// K32): also each (token, block)'s sum.  VEC: 16-byte aligned rows.
template <bool K32, bool SUMS, bool VEC>
__global__ __launch_bounds__(256) void mm_split_x(const float* __restrict__ x, uint32_t n, uint32_t ldx, uint32_t K,
                                                  uint32_t ntt, uint32_t nblk, __bf16* __restrict__ planes,
                                                  float* __restrict__ sums) {
  const uint32_t lane = threadIdx.x & 63u, item = blockIdx.x * 4u + (threadIdx.x >> 6);
  if (item >= ntt * nblk) return;
  const uint32_t tt = item % ntt, blk = item / ntt;
  uint4* out = reinterpret_cast<uint4*>(planes) + lane;
  float sum = 0.f;
#pragma unroll
  for (uint32_t h = 0; h < 2; ++h) {
    const uint32_t t = tt * 32u + (K32 ? 16u * h + (lane & 15u) : lane & 31u);
    const uint32_t k = 32u * blk + (K32 ? 8u * (lane >> 4) : 16u * h + 8u * (lane >> 5));
    float e[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (t < n && k < K) {
      const float* p = x + (size_t)t * ldx + k;
      if constexpr (VEC) {
        const float4 v0 = reinterpret_cast<const float4*>(p)[0], v1 = reinterpret_cast<const float4*>(p)[1];
        e[0] = v0.x; e[1] = v0.y; e[2] = v0.z; e[3] = v0.w;
        e[4] = v1.x; e[5] = v1.y; e[6] = v1.z; e[7] = v1.w;
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = p[i];
      }
    }
    uint32_t pc[3][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      sum += e[i];
      e[i] = __uint_as_float(__float_as_uint(e[i]) ^ (blk << 31));
      const uint32_t hi = __float_as_uint(e[i]) & 0xFFFF0000u;
      const float r1 = e[i] - __uint_as_float(hi);  // exact
      const uint32_t mid = __float_as_uint(r1) & 0xFFFF0000u;
      pc[0][i] = hi;
      pc[1][i] = mid;
      pc[2][i] = __float_as_uint(r1 - __uint_as_float(mid));  // exact, at most 8 significant bits
    }
#pragma unroll
    for (uint32_t p = 0; p < 3; ++p) {
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = __builtin_amdgcn_perm(pc[p][2 * i + 1], pc[p][2 * i], 0x07060302u);
      out[((size_t)(2u * blk + h) * ntt + tt) * 192u + p * 64u] = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  if constexpr (SUMS) {
    sum += __shfl_xor(sum, 32);
    if (lane < 32u) sums[(size_t)(blk * ntt + tt) * 32u + lane] = sum;
  }
}

// ------------------------------------------------------------------ host side

namespace {
constexpr uint64_t al64(uint64_t v) { return (v + 63) / 64 * 64; }

// Token tiles a workgroup takes (three or more tiles: launches of more than 64
// tokens): four where that pads at most one tile, or in launches of more than
// eight (nine to sixteen: at most three tiles of padding), else two.
uint32_t gt_wm(uint64_t ntt) {
  return ntt % 4 == 0 || ntt % 4 == 3 || ntt > 8 ? 4u : 2u;
}

struct GtShape {
  uint32_t ntt, wm, mtiles, nstages, spp, nsplit;
};
GtShape gt_shape(uint64_t groups, uint64_t mtot, uint64_t K, uint64_t n) {  // the same for all n of one tile count
  GtShape g{};
  g.ntt = (uint32_t)((n + 31) / 32);
  g.wm = gt_wm(g.ntt);
  g.mtiles = (g.ntt + g.wm - 1) / g.wm;
  g.nstages = (uint32_t)((K + 63) / 64);
  // Splits: the cheapest by a simple count, in stages of one workgroup.
  const uint64_t tiles = groups * g.mtiles;
  double best = 1e30;
  for (uint32_t sp = 1; sp <= g.nstages / 4 || sp == 1; ++sp) {
    const uint64_t spp = (g.nstages + sp - 1) / sp, eff = (g.nstages + spp - 1) / spp, w = tiles * eff;
    // two workgroups fit a CU and take 4 / 3 of one's time
    const uint64_t full = w / 512, rest = w % 512;
    const double units = 2.0 * full + (rest == 0 ? 0.0 : rest <= 256 ? 1.5 : 2.0);
    const double cost = units * (spp + 3) + (double)eff * g.ntt * 32 * mtot * 8.0 / (4.5e12 * 2.76e-6);
    if (cost < best * 0.97) {
      best = cost;
      g.spp = (uint32_t)spp;
      g.nsplit = (uint32_t)eff;
    }
  }
  return g;
}
uint64_t gt_plane_floats(uint64_t ntt, uint64_t nstages) { return al64(nstages * 4 * ntt * 192 * 4); }
uint64_t gt_sum_floats(uint64_t ntt, uint64_t nstages) { return al64(nstages * 2 * ntt * 32); }
}  // namespace

uint64_t mm_tile_ws_floats(uint64_t groups, uint64_t mtot, uint64_t K, uint64_t n) {
  const GtShape g = gt_shape(groups, mtot, K, n);
  return gt_plane_floats(g.ntt, g.nstages) + gt_sum_floats(g.ntt, g.nstages) + (uint64_t)g.nsplit * n * mtot;
}

template <uint32_t T>
static void launch_tile_t(const GtArgs& a, uint32_t wm, uint32_t grid, hipStream_t st) {
  if (wm == 2) RF_KLAUNCH((mm_tile<T, 2>), dim3(grid), dim3(GT_THREADS), 0, st, a);
  else RF_KLAUNCH((mm_tile<T, 4>), dim3(grid), dim3(GT_THREADS), 0, st, a);
}

hipError_t launch_mm_tile(uint32_t t, const MmTileSeg* segs, int nseg, const float* x, uint64_t ldx, uint64_t n,
                          uint64_t K, float* ws, uint64_t ws_floats, hipStream_t st, MmTileOut* out) {
  GtArgs a{};
  uint64_t groups = 0, mtot = 0;
  const int nreg = t == T_Q6_K ? 4 : 2;
  for (int i = 0; i < nseg; ++i) {
    for (int k = 0; k < nreg; ++k) {
      a.seg[i].reg[k] = segs[i].reg[k];
      a.seg[i].bytes[k] = segs[i].bytes[k];
    }
    a.seg[i].rows = (uint32_t)segs[i].rows;
    a.seg[i].group_begin = (uint32_t)groups;
    a.seg[i].col = (uint32_t)mtot;
    groups += (segs[i].rows + GT_ROWS - 1) / GT_ROWS;
    mtot += segs[i].rows;
  }
  const GtShape g = gt_shape(groups, mtot, K, n);
  if (mm_tile_ws_floats(groups, mtot, K, n) > ws_floats) return hipErrorInvalidValue;
  const uint64_t grid = groups * g.mtiles * g.nsplit;
  if (grid > 0x7FFFFFFFull || (uint64_t)g.ntt * g.nstages > 0x3FFFFFFFull) return hipErrorInvalidValue;
  __bf16* planes = reinterpret_cast<__bf16*>(ws);
  float* sums = ws + gt_plane_floats(g.ntt, g.nstages);
  a.nseg = (uint32_t)nseg;
  a.n = (uint32_t)n;
  a.ntt = g.ntt;
  a.K = (uint32_t)K;
  a.nstages = g.nstages;
  a.spp = g.spp;
  a.mtot = (uint32_t)mtot;
  a.mtiles = g.mtiles;
  a.groups = (uint32_t)groups;
  a.nsplit = g.nsplit;
  a.planes = planes;
  a.sums = sums;
  a.part = sums + gt_sum_floats(g.ntt, g.nstages);
  const uint32_t nblk = 2 * g.nstages;
  const dim3 sg((g.ntt * nblk + 3) / 4);
  const bool vec = (reinterpret_cast<uintptr_t>(x) & 15u) == 0 && ldx % 4 == 0;
  auto split = t == T_Q4_K   ? (vec ? mm_split_x<false, true, true> : mm_split_x<false, true, false>)
               : t == T_Q6_K ? (vec ? mm_split_x<false, false, true> : mm_split_x<false, false, false>)
                             : (vec ? mm_split_x<true, false, true> : mm_split_x<true, false, false>);
  RF_KLAUNCH(split, sg, dim3(256), 0, st, x, a.n, (uint32_t)ldx, a.K, g.ntt, nblk, planes, sums);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  switch (t) {
    case T_Q8_0: launch_tile_t<T_Q8_0>(a, g.wm, (uint32_t)grid, st); break;
    case T_Q4_0: launch_tile_t<T_Q4_0>(a, g.wm, (uint32_t)grid, st); break;
    case T_Q4_K: launch_tile_t<T_Q4_K>(a, g.wm, (uint32_t)grid, st); break;
    default: launch_tile_t<T_Q6_K>(a, g.wm, (uint32_t)grid, st); break;
  }
  out->part = a.part;
  out->nsplit = g.nsplit;
  return hipGetLastError();
}

hipError_t load_module_gemm() {
  hipFuncAttributes fa;
  return hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(mm_split_x<true, false, true>));
}

}  // namespace rf
