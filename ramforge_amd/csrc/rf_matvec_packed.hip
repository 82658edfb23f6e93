// rf_matvec_packed.hip — batch-1 matvec on the device-native ("packed")
// layout of Q8_0, Q4_0, Q4_K and Q6_K matrices (gfx950).
//
// Same arithmetic as quant::matvec_q8_0 / matvec_q4_0 / matvec_q4_k /
// matvec_q6_k (core/src/quant.rs:898-1327): y[o] = sum over blocks of the
// block's decoded weights times x, with the reference's codes and scales;
// only the memory layout differs.
//
// Packed layout of a [rows][in] matrix: the bytes of every block are split
// into regions, each stored for all rows, row-major (same byte count as the
// GGUF payload):
//   Q8_0 / Q4_0: codes (32 / 16 bytes per block; Q4_0 keeps the GGUF nibble
//                order), f16 scales (2 bytes per block)
//   Q4_K:        codes (qs, 128 bytes per block), header (d, dmin, the 12
//                6-bit scale/min bytes: 16 bytes per block)
//   Q6_K:        ql (128), qh (64), int8 scales (16), f16 d (2 per block)
// GGUF interleaves these, so its blocks are never 16-byte aligned.  Split
// apart, the code bytes of a row are one aligned stream that a wavefront reads
// with 16-byte loads straight into registers.
//
// Work decomposition: lane l of a wavefront owns bytes [1024c + 16l, +16) of
// "chunk" c of a row's codes (16 Q8_0 codes, or 32 codes of the 4-/6-bit
// formats); one 16-byte load per lane moves 1 KiB per instruction.  The 16
// or 32 weights of a lane meet one or two 16-element "units" of x: Q4_0's low
// nibbles are elements j, its high nibbles j + 16; Q4_K's are 32 apart (two
// sub-blocks of a 64-element group); Q6_K's 64 apart.  x (times the norm
// weights when the RMSNorm prologue is fused) and the sum of every unit are
// staged in LDS once per workgroup, so no register holds x between steps.  A
// wavefront owns U whole rows (every chunk), so no partial sum crosses
// wavefronts and the main loop has no barrier; a step is U rows x LPW chunks
// and the next step's codes are requested before the current one is decoded
// (NB register buffers).  Row sums are DPP row reductions plus readlane.
// Fusions as in rf_matvec.hip: RMSNorm prologue, residual or SiLU(gate)*up
// epilogue, up to three output segments.
#include "rf_kernels.h"

#include <algorithm>
#include <cstdio>
#include <mutex>
#include <type_traits>

namespace rf {

typedef uint32_t nv_u32x4 __attribute__((ext_vector_type(4)));

// Tasks (row groups) per wavefront whose residual is staged in LDS.
constexpr uint32_t PK_RES_SLOTS = 8;
// Word 3 of a raw (untyped, stride 0) buffer resource on gfx9-family parts,
// and the cache-policy operand of a streaming (nt) load.
constexpr int PK_RSRC_WORD3 = 0x00020000;
constexpr int PK_AUX_NT = 2;
// Upper bound of the kernel's static LDS (norm partials and staged
// residuals: 16 + 16 * PK_RES_SLOTS floats at 1024 threads).
constexpr uint64_t PK_STATIC_LDS = 1024;

typedef __amdgpu_buffer_rsrc_t PkRsrc;

// ---------------------------------------------------------------- formats
//
// PkFmt<T>:
//   QK, EPB      block elements, elements per byte of the code region
//   NREG         regions; row_bytes(k, in) = bytes of region k per row
//   Meta         what a lane loads besides its 16 code bytes
//   fetch        loads of one lane at code byte b of the row
//   code         the lane's code word i (0 .. 3)
//   unit_elem    first element of unit h of the lane whose codes start at b
//   word         decode code word i against x words (units 0 and 1)
//   finish       scale the unit sums into the chunk's contribution
//   INTX         codes are summed against x's int8 digit planes (idot,
//                ifinish) instead of decoded to float (word, finish)
// Lane constants (which sub-block / half a lane's 16 bytes fall in) depend
// only on b % 128 = 16 (lane % 8), because every chunk starts at a multiple of
// 1024 bytes.

template <uint32_t T> struct PkFmt;

// x digits of one unit (matvec_packed's prologue): x = s X with the int32
// X = 2^24 a + 2^16 b + 2^8 c + e in balanced int8 digits (PK_PLANES planes);
// S[p] = sum of codes times digit plane p, exact in int32 (|S| < 2^18).  The
// unit's value is s times S[0] 2^24 + S[1] 2^16 + S[2] 2^8 + S[3]: the pairs
// are joined exactly in int32 (|S[0] 2^8 + S[1]| < 2^26), then two
// conversions and one fma round, each at most 2^-24 relative.
constexpr int PK_PLANES = 4;
__device__ __forceinline__ float pk_digits(const int* S) {
  const int hi = S[0] * 256 + S[1], lo = S[2] * 256 + S[3];
  return fmaf((float)hi, 65536.f, (float)lo);
}

// Non-finite x (matvec_packed's fallback): the kind of the reference's
// term deq * x, as bit 0 NaN, bit 1 +inf, bit 2 -inf.
__device__ __forceinline__ uint32_t pk_term_kind(float deq, float x) {
  const float t = deq * x;
  return t != t ? 1u : (t == __builtin_inff() ? 2u : (t == -__builtin_inff() ? 4u : 0u));
}
__device__ __forceinline__ uint32_t pk_word_kinds(const float* deq, const float4& x) {
  return pk_term_kind(deq[0], x.x) | pk_term_kind(deq[1], x.y) | pk_term_kind(deq[2], x.z) |
         pk_term_kind(deq[3], x.w);
}

template <> struct PkFmt<T_Q8_0> {
  static constexpr uint32_t QK = 32, EPB = 1, NREG = 2;
  static constexpr bool INTX = true;
  __host__ __device__ static uint64_t row_bytes(int k, uint64_t in) { return k == 0 ? in : in / 32 * 2; }
  typedef uint32_t Meta;  // f16 scale bits
  struct Lane {
    __device__ explicit Lane(uint32_t) {}
  };
  __device__ static void fetch(nv_u32x4& q, Meta& m, const PkRsrc* r, uint32_t b) {
    q = __builtin_amdgcn_raw_buffer_load_b128(r[0], b, 0, PK_AUX_NT);
    m = __builtin_amdgcn_raw_buffer_load_b16(r[1], (b >> 5) << 1, 0, 0);  // block b/32, 2 bytes each
  }
  __device__ static uint32_t code(const Lane&, const nv_u32x4& q, const Meta&, int i) { return q[i]; }
  __device__ static uint32_t unit_elem(uint32_t b, uint32_t) { return b; }
  // signed codes times x, each product exact up to its own rounding (a zero
  // code adds exactly nothing, as the reference's (q * d) * x does)
  __device__ static void word(const Lane&, uint32_t q, const Meta&, int, const float4& xv, const float4&,
                              float& s0, float&) {
    s0 = fmaf(rf_sb(q, 0), xv.x, s0); s0 = fmaf(rf_sb(q, 1), xv.y, s0);
    s0 = fmaf(rf_sb(q, 2), xv.z, s0); s0 = fmaf(rf_sb(q, 3), xv.w, s0);
  }
  __device__ static float finish(const Lane&, const nv_u32x4&, const Meta& m, float s0, float, float, float) {
    return rf_half_to_float_fast(m) * s0;
  }
  // the codes are signed bytes: one dot4 per word and digit plane
  __device__ static void idot(const Lane&, const nv_u32x4& q, const nv_u32x4* P, int (*S)[PK_PLANES]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int p = 0; p < PK_PLANES; ++p)
        S[0][p] = __builtin_amdgcn_sdot4((int)q[i], (int)P[p][i], S[0][p], false);
  }
  __device__ static float ifinish(const Lane&, const Meta& m, int (*S)[PK_PLANES], const float2* u) {
    return rf_half_to_float_fast(m) * (u[0].x * pk_digits(S[0]));
  }
  // word i's terms, each weight decoded as the reference does (quant.rs:177-181: q * d)
  __device__ static uint32_t kinds(const Lane&, uint32_t q, const Meta& m, int, const float4& xv, const float4&) {
    const float d = rf_half_to_float_fast(m);
    float deq[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) deq[k] = (float)(int8_t)((q >> (8 * k)) & 0xFFu) * d;
    return pk_word_kinds(deq, xv);
  }
};

template <> struct PkFmt<T_Q4_0> {
  static constexpr uint32_t QK = 32, EPB = 2, NREG = 2;
  static constexpr bool INTX = true;
  __host__ __device__ static uint64_t row_bytes(int k, uint64_t in) { return k == 0 ? in / 2 : in / 32 * 2; }
  typedef uint32_t Meta;
  struct Lane {
    __device__ explicit Lane(uint32_t) {}
  };
  __device__ static void fetch(nv_u32x4& q, Meta& m, const PkRsrc* r, uint32_t b) {
    q = __builtin_amdgcn_raw_buffer_load_b128(r[0], b, 0, PK_AUX_NT);
    m = __builtin_amdgcn_raw_buffer_load_b16(r[1], (b >> 4) << 1, 0, 0);  // block b/16
  }
  template <class M>
  __device__ static uint32_t code(const Lane&, const nv_u32x4& q, const M&, int i) { return q[i]; }
  // byte j: low nibble -> element j, high nibble -> element j + 16 (quant.rs:84-113)
  __device__ static uint32_t unit_elem(uint32_t b, uint32_t h) { return 2u * b + 16u * h; }
  // The signed codes nibble - 8 as int8 bytes 16 (nibble - 8): products with
  // x are exact up to their own rounding (no -8 sum(x) correction to cancel
  // against), and the factor 16 comes off exactly in finish.  (Converting
  // each nibble with v_cvt_off_f32_i4 instead, (nibble ^ 8) / 16 with the
  // byte picked by SDWA, saves two instructions per word but timed the same:
  // 14336 x 4096 9.52 against 9.47 us, 4096 x 14336 10.60 against 10.56.)
  __device__ static void word(const Lane&, uint32_t q, const Meta&, int, const float4& xv, const float4& xw,
                              float& s0, float& s1) {
    const uint32_t lo = rf_opaque(rf_top_signed(q, 4)), hi = rf_opaque(rf_top_signed(q >> 4, 4));
    s0 = fmaf(rf_sb(lo, 0), xv.x, s0); s0 = fmaf(rf_sb(lo, 1), xv.y, s0);
    s0 = fmaf(rf_sb(lo, 2), xv.z, s0); s0 = fmaf(rf_sb(lo, 3), xv.w, s0);
    s1 = fmaf(rf_sb(hi, 0), xw.x, s1); s1 = fmaf(rf_sb(hi, 1), xw.y, s1);
    s1 = fmaf(rf_sb(hi, 2), xw.z, s1); s1 = fmaf(rf_sb(hi, 3), xw.w, s1);
  }
  __device__ static float finish(const Lane&, const nv_u32x4&, const Meta& m, float s0, float s1, float, float) {
    return rf_half_to_float_fast(m) * ((s0 + s1) * 0.0625f);
  }
  // the same int8 bytes 16 (nibble - 8) against the digits: exact int32 sums
  __device__ static void idot(const Lane&, const nv_u32x4& q, const nv_u32x4* P, int (*S)[PK_PLANES]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t lo = rf_opaque(rf_top_signed(q[i], 4)), hi = rf_opaque(rf_top_signed(q[i] >> 4, 4));
#pragma unroll
      for (int p = 0; p < PK_PLANES; ++p) {
        S[0][p] = __builtin_amdgcn_sdot4((int)lo, (int)P[p][i], S[0][p], false);
        S[1][p] = __builtin_amdgcn_sdot4((int)hi, (int)P[PK_PLANES + p][i], S[1][p], false);
      }
    }
  }
  __device__ static float ifinish(const Lane&, const Meta& m, int (*S)[PK_PLANES], const float2* u) {
    const float s = fmaf(u[0].x, pk_digits(S[0]), u[1].x * pk_digits(S[1]));
    return rf_half_to_float_fast(m) * (s * 0.0625f);
  }
  // (nibble - 8) * d, low nibbles against unit 0, high against unit 1 (quant.rs:104-112)
  __device__ static uint32_t kinds(const Lane&, uint32_t q, const Meta& m, int, const float4& xv, const float4& xw) {
    const float d = rf_half_to_float_fast(m);
    float lo[4], hi[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      lo[k] = (float)((int)((q >> (8 * k)) & 0xFu) - 8) * d;
      hi[k] = (float)((int)((q >> (8 * k + 4)) & 0xFu) - 8) * d;
    }
    return pk_word_kinds(lo, xv) | pk_word_kinds(hi, xw);
  }
};

// Q4_K (quant.rs:186-255): a 256-element block is 4 groups of 64; byte l of
// group g holds element 64g + l (low nibble, sub-block 2g) and 64g + 32 + l
// (high nibble, sub-block 2g + 1).  A lane's 16 bytes are half hh of group g
// (g = (lane % 8) / 2, hh = lane % 2).  Sub-block j has 6-bit scale and min
// per get_scale_min (quant.rs:216-226); value d*sc*q - dmin*m.
template <> struct PkFmt<T_Q4_K> {
  static constexpr uint32_t QK = 256, EPB = 2, NREG = 2;
  static constexpr bool INTX = false;
  __host__ __device__ static uint64_t row_bytes(int k, uint64_t in) { return k == 0 ? in / 2 : in / 256 * 16; }
  typedef nv_u32x4 Meta;  // d | dmin << 16, then scale bytes 0-3, 4-7, 8-11
  struct Lane {
    uint32_t sh;  // bit offset of sub-block 2g's byte in its scale word
    bool hi;      // g >= 2: the 4+2-bit form
    __device__ explicit Lane(uint32_t lane) {
      const uint32_t g = (lane & 7u) >> 1;
      sh = 16u * (g & 1u);
      hi = g >= 2u;
    }
  };
  __device__ static void fetch(nv_u32x4& q, Meta& m, const PkRsrc* r, uint32_t b) {
    q = __builtin_amdgcn_raw_buffer_load_b128(r[0], b, 0, PK_AUX_NT);
    m = __builtin_amdgcn_raw_buffer_load_b128(r[1], (b >> 7) << 4, 0, 0);
  }
  template <class M>
  __device__ static uint32_t code(const Lane&, const nv_u32x4& q, const M&, int i) { return q[i]; }
  __device__ static uint32_t unit_elem(uint32_t b, uint32_t h) {
    const uint32_t o = b & 127u;
    return (b >> 7) * 256u + 64u * (o >> 5) + 16u * ((o >> 4) & 1u) + 32u * h;
  }
  // unsigned nibbles: the min term dmin * m * sum(x) is part of the format
  __device__ static void word(const Lane&, uint32_t q, const Meta&, int, const float4& xv, const float4& xw,
                              float& s0, float& s1) {
    const uint32_t lo = rf_opaque(q & 0x0F0F0F0Fu), hi = rf_opaque((q >> 4) & 0x0F0F0F0Fu);
    s0 = fmaf(rf_ub(lo, 0), xv.x, s0); s0 = fmaf(rf_ub(lo, 1), xv.y, s0);
    s0 = fmaf(rf_ub(lo, 2), xv.z, s0); s0 = fmaf(rf_ub(lo, 3), xv.w, s0);
    s1 = fmaf(rf_ub(hi, 0), xw.x, s1); s1 = fmaf(rf_ub(hi, 1), xw.y, s1);
    s1 = fmaf(rf_ub(hi, 2), xw.z, s1); s1 = fmaf(rf_ub(hi, 3), xw.w, s1);
  }
  __device__ static float finish(const Lane& L, const nv_u32x4&, const Meta& m, float s0, float s1, float xs0, float xs1) {
    // sub-blocks j = 2g (+0) and 2g + 1 (+8 bits): for j < 4 sc = S[j] & 63,
    // m = S[j+4] & 63; else sc = (S[j+4] & 15) | (S[j-4] >> 6) << 4,
    // m = (S[j+4] >> 4) | (S[j] >> 6) << 4  (S = the 12 scale bytes)
    uint32_t sc[2], mn[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t s = L.sh + 8u * k;
      const uint32_t a = (m.y >> s) & 0xFFu, c = (m.z >> s) & 0xFFu, e = (m.w >> s) & 0xFFu;
      sc[k] = L.hi ? ((e & 15u) | ((a >> 6) << 4)) : (a & 63u);
      mn[k] = L.hi ? ((e >> 4) | ((c >> 6) << 4)) : (c & 63u);
    }
    const float d = rf_half_to_float_fast(m.x & 0xFFFFu), dmin = rf_half_to_float_fast(m.x >> 16);
    const float r0 = fmaf(d * (float)sc[0], s0, -(dmin * (float)mn[0]) * xs0);
    return fmaf(d * (float)sc[1], s1, fmaf(-(dmin * (float)mn[1]), xs1, r0));
  }
  // d * sc and dmin * m of sub-block 2g + h
  __device__ static void scale_min(const Lane& L, const Meta& m, int h, float& d1, float& m1) {
    const float d = rf_half_to_float_fast(m.x & 0xFFFFu), dmin = rf_half_to_float_fast(m.x >> 16);
    const uint32_t s = L.sh + 8u * h;
    const uint32_t a = (m.y >> s) & 0xFFu, c = (m.z >> s) & 0xFFu, e = (m.w >> s) & 0xFFu;
    d1 = d * (float)(L.hi ? ((e & 15u) | ((a >> 6) << 4)) : (a & 63u));
    m1 = dmin * (float)(L.hi ? ((e >> 4) | ((c >> 6) << 4)) : (c & 63u));
  }
  // d1 * q - m1 with d1 = d * sc, m1 = dmin * m (quant.rs:228-254), no fused multiply-add
  __device__ static uint32_t kinds(const Lane& L, uint32_t q, const Meta& m, int, const float4& xv, const float4& xw) {
    uint32_t out = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float d1, m1, deq[4];
      scale_min(L, m, h, d1, m1);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float prod = d1 * (float)((q >> (8 * k + 4 * h)) & 0xFu);
        deq[k] = __fsub_rn(prod, m1);
      }
      out |= pk_word_kinds(deq, h ? xw : xv);
    }
    return out;
  }
};

// Q6_K (quant.rs:347-407): per 128-element half hf, byte r < 64 of ql holds
// element 128hf + r (low nibble) and 128hf + 64 + r (high nibble); their two
// high bits are bits 2k and 2k + 4 of qh[32hf + r % 32], k = r / 32; scales
// sc[8hf + 2k + (r % 32) / 16] and the same + 4; value d*sc*(q - 32).  A
// lane's 16 bytes sit at r = 16 (lane % 4) of half hf = (lane % 8) / 4.
template <> struct PkFmt<T_Q6_K> {
  static constexpr uint32_t QK = 256, EPB = 2, NREG = 4;
  static constexpr bool INTX = false;
  __host__ __device__ static uint64_t row_bytes(int k, uint64_t in) {
    return k == 0 ? in / 2 : k == 1 ? in / 4 : k == 2 ? in / 256 * 16 : in / 256 * 2;
  }
  struct Meta {
    nv_u32x4 qh, sc;
    uint32_t d;
  };
  struct Lane {
    uint32_t qsh;  // 2k: shift of the low unit's high bits
    uint32_t bsh;  // bit offset of the low unit's scale byte in its word
    bool hf;       // half 1: scale words 2 and 3 instead of 0 and 1
    __device__ explicit Lane(uint32_t lane) {
      qsh = 2u * ((lane & 3u) >> 1);
      bsh = 8u * (qsh + (lane & 1u));
      hf = (lane & 4u) != 0;
    }
  };
  __device__ static void fetch(nv_u32x4& q, Meta& m, const PkRsrc* r, uint32_t b) {
    const uint32_t blk = b >> 7, o = b & 127u;
    q = __builtin_amdgcn_raw_buffer_load_b128(r[0], b, 0, PK_AUX_NT);
    m.qh = __builtin_amdgcn_raw_buffer_load_b128(r[1], blk * 64u + 32u * (o >> 6) + (o & 31u), 0, PK_AUX_NT);
    m.sc = __builtin_amdgcn_raw_buffer_load_b128(r[2], blk * 16u, 0, 0);
    m.d = __builtin_amdgcn_raw_buffer_load_b16(r[3], blk * 2u, 0, 0);
  }
  __device__ static uint32_t code(const Lane&, const nv_u32x4& q, const Meta&, int i) { return q[i]; }
  __device__ static uint32_t unit_elem(uint32_t b, uint32_t h) {
    const uint32_t o = b & 127u;
    return (b >> 7) * 256u + 128u * (o >> 6) + (o & 63u) + 64u * h;
  }
  __device__ static void word(const Lane& L, uint32_t q, const Meta& m, int i, const float4& xv, const float4& xw,
                              float& s0, float& s1) {
    // the 6-bit codes q - 32 as int8 bytes 4 (q - 32): exact products, the
    // factor 4 comes off exactly in finish
    const uint32_t h = m.qh[i];
    const uint32_t lo = rf_opaque(rf_top_signed((q & 0x0F0F0F0Fu) | (((h >> L.qsh) & 0x03030303u) << 4), 6));
    const uint32_t hi =
        rf_opaque(rf_top_signed(((q >> 4) & 0x0F0F0F0Fu) | (((h >> (L.qsh + 4u)) & 0x03030303u) << 4), 6));
    s0 = fmaf(rf_sb(lo, 0), xv.x, s0); s0 = fmaf(rf_sb(lo, 1), xv.y, s0);
    s0 = fmaf(rf_sb(lo, 2), xv.z, s0); s0 = fmaf(rf_sb(lo, 3), xv.w, s0);
    s1 = fmaf(rf_sb(hi, 0), xw.x, s1); s1 = fmaf(rf_sb(hi, 1), xw.y, s1);
    s1 = fmaf(rf_sb(hi, 2), xw.z, s1); s1 = fmaf(rf_sb(hi, 3), xw.w, s1);
  }
  __device__ static float finish(const Lane& L, const nv_u32x4&, const Meta& m, float s0, float s1, float, float) {
    const uint32_t w0 = L.hf ? m.sc.z : m.sc.x, w1 = L.hf ? m.sc.w : m.sc.y;
    const float sc0 = (float)(int32_t)(int8_t)((w0 >> L.bsh) & 0xFFu);
    const float sc1 = (float)(int32_t)(int8_t)((w1 >> L.bsh) & 0xFFu);
    const float d = rf_half_to_float_fast(m.d);
    return d * (fmaf(sc0, s0, sc1 * s1) * 0.25f);
  }
  // (d * sc) * (q - 32) (quant.rs:376-406)
  __device__ static uint32_t kinds(const Lane& L, uint32_t q, const Meta& m, int i, const float4& xv,
                                   const float4& xw) {
    const uint32_t h = m.qh[i];
    const uint32_t w0 = L.hf ? m.sc.z : m.sc.x, w1 = L.hf ? m.sc.w : m.sc.y;
    const float d = rf_half_to_float_fast(m.d);
    const float ds0 = d * (float)(int32_t)(int8_t)((w0 >> L.bsh) & 0xFFu);
    const float ds1 = d * (float)(int32_t)(int8_t)((w1 >> L.bsh) & 0xFFu);
    float lo[4], hi[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t sh = 8u * k;
      const int ql = (int)(((q >> sh) & 0xFu) | (((h >> (L.qsh + sh)) & 3u) << 4));
      const int qh = (int)(((q >> (sh + 4u)) & 0xFu) | (((h >> (L.qsh + 4u + sh)) & 3u) << 4));
      lo[k] = ds0 * (float)(ql - 32);
      hi[k] = ds1 * (float)(qh - 32);
    }
    return pk_word_kinds(lo, xv) | pk_word_kinds(hi, xw);
  }
};

// The same decodes on the GGUF payload itself (T | PK_GGUF): one region, the
// rows as stored, a lane's code bytes found inside the blocks instead of in
// the code stream.  Blocks of 18, 22, 34 and 210 bytes put the 16-byte loads
// on any even address, which the parts take in the unaligned access mode the
// HSA runtime sets; 64 lanes still cover one contiguous span of blocks.
// Against the kernels this replaces (wavefront- or tile-staged: each byte
// through LDS both ways), eager calls: Q8_0 4096 x 4096 6.6 -> 5.5 us, 4096 x
// 14336 16.3 -> 12.3; Q4_0 14336 x 4096 11.0 -> 8.9; Q5_0 19.6 -> 10.4; Q4_K
// 14.0 -> 9.1, 4096 x 14336 18.8 -> 10.8; Q5_K 14336 x 4096 21.5 -> 11.0;
// Q6_K 16.2 -> 11.9, 128256 x 4096 114 -> 92.  Non-temporal loads, which suit
// the packed regions, are slower here (Q8_0 14336 x 4096 14.1): neighbouring
// loads share cache lines.
constexpr uint32_t PK_GGUF = 0x100;
__host__ __device__ constexpr uint32_t pk_base(uint32_t t) { return t & 0xFFu; }

template <> struct PkFmt<T_Q8_0 | PK_GGUF> : PkFmt<T_Q8_0> {
  static constexpr uint32_t NREG = 1;
  static constexpr bool INTX = false;
  __host__ __device__ static uint64_t row_bytes(int, uint64_t in) { return in / 32 * 34; }
  __device__ static void fetch(nv_u32x4& q, Meta& m, const PkRsrc* r, uint32_t b) {
    const uint32_t o = (b >> 5) * 34u;
    q = __builtin_amdgcn_raw_buffer_load_b128(r[0], o + 2u + (b & 31u), 0, 0);
    m = __builtin_amdgcn_raw_buffer_load_b16(r[0], o, 0, 0);
  }
};
template <> struct PkFmt<T_Q4_0 | PK_GGUF> : PkFmt<T_Q4_0> {
  static constexpr uint32_t NREG = 1;
  static constexpr bool INTX = false;
  __host__ __device__ static uint64_t row_bytes(int, uint64_t in) { return in / 32 * 18; }
  __device__ static void fetch(nv_u32x4& q, Meta& m, const PkRsrc* r, uint32_t b) {
    const uint32_t o = (b >> 4) * 18u;
    q = __builtin_amdgcn_raw_buffer_load_b128(r[0], o + 2u, 0, 0);
    m = __builtin_amdgcn_raw_buffer_load_b16(r[0], o, 0, 0);
  }
};
template <> struct PkFmt<T_Q4_K | PK_GGUF> : PkFmt<T_Q4_K> {
  static constexpr uint32_t NREG = 1;
  __host__ __device__ static uint64_t row_bytes(int, uint64_t in) { return in / 256 * 144; }
  __device__ static void fetch(nv_u32x4& q, Meta& m, const PkRsrc* r, uint32_t b) {
    const uint32_t o = (b >> 7) * 144u;
    q = __builtin_amdgcn_raw_buffer_load_b128(r[0], o + 16u + (b & 127u), 0, 0);
    m = __builtin_amdgcn_raw_buffer_load_b128(r[0], o, 0, 0);
  }
};
template <> struct PkFmt<T_Q6_K | PK_GGUF> : PkFmt<T_Q6_K> {
  static constexpr uint32_t NREG = 1;
  __host__ __device__ static uint64_t row_bytes(int, uint64_t in) { return in / 256 * 210; }
  __device__ static void fetch(nv_u32x4& q, Meta& m, const PkRsrc* r, uint32_t b) {
    const uint32_t base = (b >> 7) * 210u, o = b & 127u;
    q = __builtin_amdgcn_raw_buffer_load_b128(r[0], base + o, 0, 0);
    m.qh = __builtin_amdgcn_raw_buffer_load_b128(r[0], base + 128u + 32u * (o >> 6) + (o & 31u), 0, 0);
    m.sc = __builtin_amdgcn_raw_buffer_load_b128(r[0], base + 192u, 0, 0);
    m.d = __builtin_amdgcn_raw_buffer_load_b16(r[0], base + 208u, 0, 0);
  }
};
// Q5_0 (quant.rs:117-151): d, qh (bit e of element e), 16 bytes of nibbles; a
// lane's 16 bytes are one block, as in Q4_0.
template <> struct PkFmt<T_Q5_0 | PK_GGUF> : PkFmt<T_Q4_0 | PK_GGUF> {
  struct Meta {
    uint32_t d, qh;
  };
  __host__ __device__ static uint64_t row_bytes(int, uint64_t in) { return in / 32 * 22; }
  __device__ static void fetch(nv_u32x4& q, Meta& m, const PkRsrc* r, uint32_t b) {
    const uint32_t o = (b >> 4) * 22u;
    q = __builtin_amdgcn_raw_buffer_load_b128(r[0], o + 6u, 0, 0);
    m.qh = __builtin_amdgcn_raw_buffer_load_b32(r[0], o + 2u, 0, 0);
    m.d = __builtin_amdgcn_raw_buffer_load_b16(r[0], o, 0, 0);
  }
  // bits 4 i .. 4 i + 3 of h as bit 4 of four bytes
  __device__ static uint32_t spread(uint32_t h, int i) {
    return ((((h >> (4 * i)) & 0xFu) * 0x00204081u) & 0x01010101u) << 4;
  }
  // the codes q - 16 as int8 bytes 8 (q - 16), the factor 8 off in finish
  __device__ static void word(const Lane&, uint32_t q, const Meta& m, int i, const float4& xv, const float4& xw,
                              float& s0, float& s1) {
    const uint32_t lo = rf_opaque(rf_top_signed((q & 0x0F0F0F0Fu) | spread(m.qh, i), 5));
    const uint32_t hi = rf_opaque(rf_top_signed(((q >> 4) & 0x0F0F0F0Fu) | spread(m.qh >> 16, i), 5));
    s0 = fmaf(rf_sb(lo, 0), xv.x, s0); s0 = fmaf(rf_sb(lo, 1), xv.y, s0);
    s0 = fmaf(rf_sb(lo, 2), xv.z, s0); s0 = fmaf(rf_sb(lo, 3), xv.w, s0);
    s1 = fmaf(rf_sb(hi, 0), xw.x, s1); s1 = fmaf(rf_sb(hi, 1), xw.y, s1);
    s1 = fmaf(rf_sb(hi, 2), xw.z, s1); s1 = fmaf(rf_sb(hi, 3), xw.w, s1);
  }
  __device__ static float finish(const Lane&, const nv_u32x4&, const Meta& m, float s0, float s1, float, float) {
    return rf_half_to_float_fast(m.d) * ((s0 + s1) * 0.125f);
  }
};
// Q5_K (quant.rs:259-343): Q4_K's header, qh[32], qs[128].  Element l of
// sub-block s has its high bit in bit s of qh[8 (s / 2) + l / 8] (the
// reference's own index), so the two bytes 8 g + 2 hh, + 1 serve a lane's
// half hh of group g: byte i / 2 for word i, bit 2 g for the low nibbles'
// sub-block and 2 g + 1 for the high ones'.
template <> struct PkFmt<T_Q5_K | PK_GGUF> : PkFmt<T_Q4_K | PK_GGUF> {
  struct Meta {
    nv_u32x4 h;
    uint32_t qh;
  };
  struct Lane : PkFmt<T_Q4_K>::Lane {
    uint32_t bit;  // 2 g
    __device__ explicit Lane(uint32_t lane) : PkFmt<T_Q4_K>::Lane(lane), bit(lane & 6u) {}
  };
  __host__ __device__ static uint64_t row_bytes(int, uint64_t in) { return in / 256 * 176; }
  __device__ static void fetch(nv_u32x4& q, Meta& m, const PkRsrc* r, uint32_t b) {
    const uint32_t base = (b >> 7) * 176u, o = b & 127u;
    q = __builtin_amdgcn_raw_buffer_load_b128(r[0], base + 48u + o, 0, 0);
    m.h = __builtin_amdgcn_raw_buffer_load_b128(r[0], base, 0, 0);
    m.qh = __builtin_amdgcn_raw_buffer_load_b16(r[0], base + 16u + 8u * (o >> 5) + 2u * ((o >> 4) & 1u), 0, 0);
  }
  __device__ static uint32_t high(const Lane& L, const Meta& m, int i, int h) {
    return ((m.qh >> (8 * (i >> 1))) >> (L.bit + h)) & 1u;
  }
  __device__ static void word(const Lane& L, uint32_t q, const Meta& m, int i, const float4& xv, const float4& xw,
                              float& s0, float& s1) {
    const uint32_t lo = rf_opaque((q & 0x0F0F0F0Fu) | (high(L, m, i, 0) * 0x10101010u));
    const uint32_t hi = rf_opaque(((q >> 4) & 0x0F0F0F0Fu) | (high(L, m, i, 1) * 0x10101010u));
    s0 = fmaf(rf_ub(lo, 0), xv.x, s0); s0 = fmaf(rf_ub(lo, 1), xv.y, s0);
    s0 = fmaf(rf_ub(lo, 2), xv.z, s0); s0 = fmaf(rf_ub(lo, 3), xv.w, s0);
    s1 = fmaf(rf_ub(hi, 0), xw.x, s1); s1 = fmaf(rf_ub(hi, 1), xw.y, s1);
    s1 = fmaf(rf_ub(hi, 2), xw.z, s1); s1 = fmaf(rf_ub(hi, 3), xw.w, s1);
  }
  __device__ static float finish(const Lane& L, const nv_u32x4& q, const Meta& m, float s0, float s1, float xs0, float xs1) {
    return PkFmt<T_Q4_K>::finish(L, q, m.h, s0, s1, xs0, xs1);
  }
  __device__ static uint32_t kinds(const Lane& L, uint32_t q, const Meta& m, int i, const float4& xv, const float4& xw) {
    uint32_t out = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float d1, m1, deq[4];
      PkFmt<T_Q4_K>::scale_min(L, m.h, h, d1, m1);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float prod = d1 * (float)(((q >> (8 * k + 4 * h)) & 0xFu) | (high(L, m, i, h) << 4));
        deq[k] = __fsub_rn(prod, m1);
      }
      out |= pk_word_kinds(deq, h ? xw : xv);
    }
    return out;
  }
};

// Rows of an even number of such blocks on a dword-aligned base (T | PK_GGUF |
// PK_DWORD): a pair of blocks is whole dwords, its first block's codes start
// two bytes into one.  The loads take whole dwords and the decode realigns
// them (code(), one v_alignbyte per word): a half-aligned 16-byte load costs
// about twice an aligned one (Q8_0 128256 x 4096 134 against 99 us).
constexpr uint32_t PK_DWORD = 0x200;
__device__ __forceinline__ uint32_t pk_realign(uint32_t lo, uint32_t hi, uint32_t sh) {
  return __builtin_amdgcn_alignbyte(hi, lo, sh);
}
// Q8_0, 17 dwords a pair: four lanes take dwords 0-3, 4-7 (first block: scale,
// then codes), 9-12, 13-16 (second block's codes); dword 8, the first block's
// last codes and the second's scale, goes to all four, and the first block's
// scale and the dword its first lane lacks come from the neighbour.
template <> struct PkFmt<T_Q8_0 | PK_GGUF | PK_DWORD> : PkFmt<T_Q8_0 | PK_GGUF> {
  struct Lane {
    uint32_t sh;
    bool first;
    __device__ explicit Lane(uint32_t lane) : sh((lane & 2u) ? 0u : 2u), first((lane & 3u) == 0u) {}
  };
  __device__ static void fetch(nv_u32x4& q, Meta& m, const PkRsrc* r, uint32_t b) {
    const uint32_t o = (b >> 6) * 68u, j = (b >> 4) & 3u;
    q = __builtin_amdgcn_raw_buffer_load_b128(r[0], o + 16u * j + 4u * (j >> 1), 0, 0);
    m = __builtin_amdgcn_raw_buffer_load_b32(r[0], o + 32u, 0, 0);
  }
  // q[0] of lane 1 (0) of the quad to lane 0 (1)
  __device__ static uint32_t swap(uint32_t v) { return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xE1, 0xF, 0xF, true); }
  __device__ static uint32_t code(const Lane& L, const nv_u32x4& q, const Meta& m, int i) {
    if (i < 3) return pk_realign(q[i], q[i + 1], L.sh);  // i is a compile-time index
    const uint32_t n = swap(q[0]);  // by all lanes
    return pk_realign(q[i], L.first ? n : m, L.sh);
  }
  __device__ static void word(const Lane&, uint32_t q, const Meta&, int, const float4& xv, const float4& xw, float& s0,
                              float& s1) {
    PkFmt<T_Q8_0>::word(PkFmt<T_Q8_0>::Lane(0), q, 0u, 0, xv, xw, s0, s1);
  }
  __device__ static float finish(const Lane& L, const nv_u32x4& q, const Meta& m, float s0, float, float, float) {
    const uint32_t n = swap(q[0]);
    const uint32_t d = L.sh == 0u ? m >> 16 : (L.first ? q[0] : n) & 0xFFFFu;
    return rf_half_to_float_fast(d) * s0;
  }
};
// Q4_0, 9 dwords a pair: a lane each, dwords 0-3 and 5-8, dword 4 to both.
template <> struct PkFmt<T_Q4_0 | PK_GGUF | PK_DWORD> : PkFmt<T_Q4_0 | PK_GGUF> {
  struct Lane {
    uint32_t sh;
    __device__ explicit Lane(uint32_t lane) : sh((lane & 1u) ? 0u : 2u) {}
  };
  __device__ static void fetch(nv_u32x4& q, Meta& m, const PkRsrc* r, uint32_t b) {
    const uint32_t o = (b >> 5) * 36u;
    q = __builtin_amdgcn_raw_buffer_load_b128(r[0], o + 20u * ((b >> 4) & 1u), 0, 0);
    m = __builtin_amdgcn_raw_buffer_load_b32(r[0], o + 16u, 0, 0);
  }
  __device__ static uint32_t code(const Lane& L, const nv_u32x4& q, const Meta& m, int i) {
    return pk_realign(q[i], i < 3 ? q[i + 1] : m, L.sh);
  }
  __device__ static void word(const Lane&, uint32_t q, const Meta&, int, const float4& xv, const float4& xw, float& s0,
                              float& s1) {
    PkFmt<T_Q4_0>::word(PkFmt<T_Q4_0>::Lane(0), q, 0u, 0, xv, xw, s0, s1);
  }
  __device__ static float finish(const Lane& L, const nv_u32x4& q, const Meta& m, float s0, float s1, float, float) {
    const uint32_t d = L.sh == 0u ? m >> 16 : q[0] & 0xFFFFu;
    return rf_half_to_float_fast(d) * ((s0 + s1) * 0.0625f);
  }
};
// Q6_K: a block starts 0 or 2 bytes into a dword by its parity, a lane constant.
template <> struct PkFmt<T_Q6_K | PK_GGUF | PK_DWORD> : PkFmt<T_Q6_K | PK_GGUF> {
  struct Meta {
    nv_u32x4 qh;
    uint32_t tail, htail, sc[3], d;
  };
  struct Lane : PkFmt<T_Q6_K>::Lane {
    uint32_t sh;
    __device__ explicit Lane(uint32_t lane) : PkFmt<T_Q6_K>::Lane(lane), sh((lane & 8u) ? 2u : 0u) {}
  };
  __device__ static void fetch(nv_u32x4& q, Meta& m, const PkRsrc* r, uint32_t b) {
    const uint32_t base = (b >> 7) * 210u, o = b & 127u, ab = base & ~3u, h = ab + 128u + 32u * (o >> 6) + (o & 31u);
    q = __builtin_amdgcn_raw_buffer_load_b128(r[0], ab + o, 0, 0);
    m.tail = __builtin_amdgcn_raw_buffer_load_b32(r[0], ab + o + 16u, 0, 0);
    m.qh = __builtin_amdgcn_raw_buffer_load_b128(r[0], h, 0, 0);
    m.htail = __builtin_amdgcn_raw_buffer_load_b32(r[0], h + 16u, 0, 0);
    const auto sc = __builtin_amdgcn_raw_buffer_load_b96(r[0], ab + 192u + 8u * (o >> 6), 0, 0);
    m.sc[0] = sc[0]; m.sc[1] = sc[1]; m.sc[2] = sc[2];
    m.d = __builtin_amdgcn_raw_buffer_load_b16(r[0], base + 208u, 0, 0);
  }
  __device__ static uint32_t code(const Lane& L, const nv_u32x4& q, const Meta& m, int i) {
    return pk_realign(q[i], i < 3 ? q[i + 1] : m.tail, L.sh);
  }
  __device__ static void word(const Lane& L, uint32_t q, const Meta& m, int i, const float4& xv, const float4& xw,
                              float& s0, float& s1) {
    PkFmt<T_Q6_K>::Meta w;
    w.qh[i] = pk_realign(m.qh[i], i < 3 ? m.qh[i + 1] : m.htail, L.sh);
    PkFmt<T_Q6_K>::word(L, q, w, i, xv, xw, s0, s1);
  }
  __device__ static float finish(const Lane& L, const nv_u32x4&, const Meta& m, float s0, float s1, float, float) {
    const uint32_t w0 = pk_realign(m.sc[0], m.sc[1], L.sh), w1 = pk_realign(m.sc[1], m.sc[2], L.sh);
    return rf_half_to_float_fast(m.d) * (fmaf(rf_sb(w0 >> L.bsh, 0), s0, rf_sb(w1 >> L.bsh, 0) * s1) * 0.25f);
  }
};

// Codes and metadata of one step: U rows x LPW chunks (twice with the "up" matrix).
template <uint32_t T, int U, int LPW, bool DUAL>
struct PkStep {
  nv_u32x4 q[U][LPW], q2[DUAL ? U : 1][LPW];
  typename PkFmt<T>::Meta m[U][LPW], m2[DUAL ? U : 1][LPW];
};

// The workgroup stages x while its first steps' codes are in flight.  x sits
// in LDS permuted so that the 16-byte reads of a step are consecutive across
// lanes (no bank conflicts): element 4i + k of unit h of lane l's slice of
// chunk c (EPL = 16 or 32 elements per slice) is stored at
// c * 64 * EPL + 256 (4h + i) + 4 l + k.  NB step buffers per wavefront: NB - 1
// steps are in flight while one is decoded.  ALLF: every step of the
// wavefront (its tasks times the steps of a row at most NB) is requested
// before the prologue and none after it, so a launch makes one memory round
// trip.
//
// MRG: x is merged from single-query attention's chunk records in the
// prologue (the merge the attention's own merge kernel does, so that launch
// is saved): per head, M = max of the chunks' m, factors f_c = exp(m_c - M),
// L = sum of l_c f_c and x = (sum of f_c o_c) / L, taken as a product with
// 1 / L.  Each thread merges half a unit (8 elements) over all chunks; the
// launch sees to 2 nunit <= NT and at most 8 chunks.
template <uint32_t T, int EPI, bool NORM, int U, int LPW, int NB, int NT, bool IX, bool ALLF = false,
          bool MRG = false>
__global__ __launch_bounds__(NT) void matvec_packed(PkArgs a) {
  auto seg_of = [&](uint32_t v) -> PkSeg {
    return (a.nseg > 2 && v >= a.seg[2].row_begin) ? a.seg[2]
                                                   : ((a.nseg > 1 && v >= a.seg[1].row_begin) ? a.seg[1] : a.seg[0]);
  };
#include "rf_matvec_packed_body.inc"
}

// A plain y = W x on GGUF bytes with just its own arguments: the 350 bytes of
// PkArgs cost an eager call 0.3 us on the host.  (One body behind a device
// function that takes the arguments by reference puts them in scratch memory:
// 8B decode 34 -> 43 ms.)
struct PkPlainArgs {
  const uint8_t* w;
  const float* x;
  float* y;
  uint32_t rows_total, in_dim;
  static constexpr const float *norm_w = nullptr, *mws = nullptr;
  static constexpr int32_t *advance = nullptr, *m_pos = nullptr;
  static constexpr float eps = 0.f;
  static constexpr uint32_t m_nsplit = 0, m_qh = 0, m_hd_log2 = 0;
};
template <uint32_t T, int LPW, int NB, int NT, bool ALLF>
__global__ __launch_bounds__(NT) void matvec_gguf(PkPlainArgs a) {
  constexpr int EPI = EPI_STORE, U = 1;
  constexpr bool NORM = false, IX = false, MRG = false;
  auto seg_of = [&](uint32_t) {
    PkSeg g{};
    g.reg[0] = a.w;
    g.y = a.y;
    return g;
  };
#include "rf_matvec_packed_body.inc"
}

// GGUF blocks -> packed layout, one thread per block (install-time only).
// Block i (row-major over rows and blocks) lands at i * (region bytes per
// block) in every region.
template <uint32_t T>
__global__ __launch_bounds__(256) void pack_blocks(const uint8_t* __restrict__ raw, uint8_t* __restrict__ packed,
                                                   uint64_t nblocks) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nblocks) return;
  constexpr uint32_t BS = Fmt<T>::BS;
  const uint8_t* b = raw + i * BS;
  auto copy = [&](uint8_t* dst, const uint8_t* src, uint32_t n) {
    for (uint32_t k = 0; k < n; ++k) dst[k] = src[k];
  };
  if constexpr (T == T_Q8_0 || T == T_Q4_0) {
    constexpr uint32_t CB = BS - 2;
    copy(packed + nblocks * CB + 2 * i, b, 2);  // f16 scale
    copy(packed + i * CB, b + 2, CB);           // codes
  } else if constexpr (T == T_Q4_K) {
    copy(packed + nblocks * 128 + 16 * i, b, 16);  // d, dmin, scales[12]
    copy(packed + i * 128, b + 16, 128);           // qs
  } else {
    uint8_t* qh = packed + nblocks * 128;
    uint8_t* sc = qh + nblocks * 64;
    uint8_t* d = sc + nblocks * 16;
    copy(packed + i * 128, b, 128);  // ql
    copy(qh + i * 64, b + 128, 64);
    copy(sc + i * 16, b + 192, 16);
    copy(d + i * 2, b + 208, 2);
  }
}

// ------------------------------------------------------------------ host side

bool packed_type(uint32_t t) { return t == T_Q8_0 || t == T_Q4_0 || t == T_Q4_K || t == T_Q6_K; }

static uint32_t pk_qk(uint32_t t) { return (t == T_Q4_K || t == T_Q5_K || t == T_Q6_K) ? 256u : 32u; }
static uint32_t pk_epb(uint32_t t) { return t == T_Q8_0 ? 1u : 2u; }

// Region k of format t: bytes per row.
static uint64_t pk_row_bytes(uint32_t t, int k, uint64_t in) {
  switch (t) {
    case T_Q8_0: return PkFmt<T_Q8_0>::row_bytes(k, in);
    case T_Q4_0: return PkFmt<T_Q4_0>::row_bytes(k, in);
    case T_Q4_K: return PkFmt<T_Q4_K>::row_bytes(k, in);
    default: return PkFmt<T_Q6_K>::row_bytes(k, in);
  }
}
static int pk_nreg(uint32_t t) { return t == T_Q6_K ? 4 : 2; }

static uint32_t pk_lds_limit() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 65536;
  if (!cached[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || n < 65536)
      n = 65536;
    cached[dev] = n;
  }
  return (uint32_t)cached[dev];
}

static uint64_t pk_nchunk(uint32_t t, uint64_t in_dim) { return (in_dim / pk_epb(pk_base(t)) + 1023) / 1024; }

static PkPlan pk_plan(uint32_t t, uint64_t in_dim) {
  PkPlan p{};
  if (in_dim == 0 || in_dim % pk_qk(t) != 0 || in_dim > (1u << 24)) return p;
  const uint64_t nchunk = pk_nchunk(t, in_dim), ups = pk_epb(t), epl = 16 * ups;
  const uint64_t lds = (nchunk * 64 * epl + nchunk * 64 * ups) * 4;
  if (lds + PK_STATIC_LDS > 65536 && lds + PK_STATIC_LDS > pk_lds_limit()) return p;  // every device has 64 KiB
  p.ok = true;
  p.lds_bytes = (uint32_t)lds;
  return p;
}

PkPlan plan_packed(uint32_t t, uint64_t in_dim) { return packed_type(t) ? pk_plan(t, in_dim) : PkPlan{}; }

PkPlan plan_gguf(uint32_t t, uint64_t in_dim) {
  return packed_type(t) || t == T_Q5_0 || t == T_Q5_K ? pk_plan(t, in_dim) : PkPlan{};
}

static int pk_cu_count() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cached[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

// Resident workgroups per CU of one kernel at one LDS size; the caller keeps
// one cache per kernel (a few distinct sizes per model).  A miss runs the
// one-time setup (dynamic LDS attribute, occupancy query) and is refused (-1)
// while st is being captured.
struct PkOccCache {
  std::mutex mu;
  uint32_t keys[16];
  int vals[16];
  int n = 0;
  uint32_t attr = 0;  // dynamic LDS the kernel has been opened up to (above 64 KiB)
};
static int pk_occupancy(PkOccCache& c, const void* kern, int nt, uint32_t lds, hipStream_t st) {
  std::lock_guard<std::mutex> lock(c.mu);
  for (int i = 0; i < c.n; ++i)
    if (c.keys[i] == lds) return c.vals[i];
  if (setup_outside_capture(st) != hipSuccess) return -1;
  if (lds > 65536 && lds > c.attr) {
    if (hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) return 0;
    c.attr = lds;
  }
  int occ = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kern, nt, lds) != hipSuccess || occ < 1) occ = 1;
  if (c.n < 16) {
    c.keys[c.n] = lds;
    c.vals[c.n] = occ;
    ++c.n;
  }
  return occ;
}

// Name of the matvec_packed instance the calling thread launched (or, in a
// planning pass, would launch) last, spelled as the profiler's kernel trace
// spells it, so that a measurement can be matched to the kernel that ran.
// Each instance's name is made once (a snprintf per launch cost an eager call
// 0.4 us).
static thread_local const char* t_last_kernel = "";
template <uint32_t T, int EPI, bool NORM, int U, int LPW, int NB, int NT, bool IX, bool ALLF, bool MRG>
static void note_kernel() {
  struct Name {
    char s[128];
    Name() {
      auto b = [](bool v) { return v ? "true" : "false"; };
      snprintf(s, sizeof s, "void rf::matvec_packed<%uu, %d, %s, %d, %d, %d, %d, %s, %s, %s>(rf::PkArgs)", T, EPI, b(NORM),
               U, LPW, NB, NT, b(IX), b(ALLF), b(MRG));
    }
  };
  static const Name name;
  t_last_kernel = name.s;
}
const char* last_packed_kernel() { return t_last_kernel; }
void clear_last_packed_kernel() { t_last_kernel = ""; }

// x as digit planes on the launches with >= 24 KiB of codes per wavefront
// (1), on every Q8_0 / Q4_0 launch whose LDS holds them (2), or float x
// everywhere (0, default): rf_tune_matvec_digits.  Measured A/B on one box,
// 8B gate/up: 3 planes 21.6-21.9 us; 4 planes 22.3-22.5 us; float x
// 22.4-22.5 us.  With 4 planes the digits no longer pay, so float x, which
// is the reference's arithmetic up to summation order, is the default.
static int g_digits = 0;
void set_matvec_digits(int mode) { g_digits = mode; }
int matvec_digits() { return g_digits; }

// LDS of the digit-plane variant: PK_PLANES bytes per element and a float2
// per 16-element unit, which also holds the float layout it falls back to.
static uint64_t pk_digit_lds(uint32_t t, uint64_t in_dim) {
  const uint64_t nchunk = pk_nchunk(t, in_dim), ups = pk_epb(t);
  return nchunk * ups * (1024u * PK_PLANES) + nchunk * 64u * ups * 8u;
}

// Grid: a whole number k of workgroups per CU (a CU with one workgroup more
// than its neighbours sets the launch time), k just large enough for about
// four rows per wavefront, at most the occupancy.  Timed on the 8B and 70B
// shapes against the fullest grid (CUs x occupancy): Q/K/V 6144x4096 8.3 vs
// 9.3 us (Q8_0), 6.3 vs 7.1 us (Q4_0); Q4_0 gate/up 15.8 vs 16.8 us; the
// other shapes within 0.2 us.
// Workgroups: whole rounds of one per CU, enough for about `per` tasks per
// wavefront, at most the kernel's occupancy.  Q8_0 gate/up launches and rows
// of up to 2048 inputs aim at 2 (8B gate/up: 768 workgroups, its occupancy,
// instead of 512, 21.5 against 21.9 us back to back, decode 545 against 540
// tok/s; the d-2048 model's gate/up 8.57 against 8.69 us); the 8B's other
// launches keep 4 (with 2: Q/K/V 7.75 against 7.30 us), and so do the other
// formats' gate/up (with 2: Q4_K 17.26 / Q4_0 16.15 against 17.30 / 16.17 us,
// Q6_K 20.72 against 20.61).
static uint64_t pk_grid(uint64_t tasks, uint64_t nw, int occ, int epi, uint64_t per = 4) {
  const uint64_t cus = (uint64_t)pk_cu_count();
  const uint64_t want = (tasks + nw - 1) / nw;
  uint64_t k = (tasks + cus * nw * per - 1) / (cus * nw * per);
  if (k < 1) k = 1;
  if (k > (uint64_t)occ) k = (uint64_t)occ;
  uint64_t grid = cus * k < want ? cus * k : want;
  if (epi == EPI_RESIDUAL) {  // at most PK_RES_SLOTS tasks per wavefront (residuals staged in LDS)
    const uint64_t need = (tasks + nw * PK_RES_SLOTS - 1) / (nw * PK_RES_SLOTS);
    if (grid < need) grid = need;
  }
  return grid;
}

// The float-x kernel of a launch and its arguments: matvec_gguf for GGUF bytes.
template <uint32_t T> using PkKernelArgs = std::conditional_t<(T & PK_GGUF) != 0, PkPlainArgs, PkArgs>;
template <uint32_t T, int EPI, bool NORM, int LPW, int NB, int NT, bool ALLF>
static constexpr auto pk_kernel() {
  if constexpr ((T & PK_GGUF) != 0) return matvec_gguf<T, LPW, NB, NT, ALLF>;
  else return matvec_packed<T, EPI, NORM, 1, LPW, NB, NT, false, ALLF>;
}

template <uint32_t T, int EPI, bool NORM, int LPW, int NB, int NT>
static hipError_t launch_pk(const PkKernelArgs<T>& a, uint32_t lds, hipStream_t st) {
  constexpr int U = 1;
  static PkOccCache cache, cache_ix;  // one per kernel variant
  auto kern = pk_kernel<T, EPI, NORM, LPW, NB, NT, false>();
  const int occ = pk_occupancy(cache, reinterpret_cast<const void*>(kern), NT, lds, st);
  if (occ < 0) return hipErrorStreamCaptureUnsupported;
  if (occ < 1) return hipErrorInvalidConfiguration;
  const uint64_t tasks = (a.rows_total + U - 1) / U, nw = NT / 64;
  uint64_t grid = pk_grid(tasks, nw, occ, EPI, ((EPI == EPI_SWIGLU && T == T_Q8_0) || a.in_dim <= 2048) ? 2 : 4);
  // Q8_0 / Q4_0 take the int8 digit planes of x when a wavefront's rows hold
  // at least 24 KiB of codes: their split costs each workgroup a longer
  // prologue, which the cheaper decode repays only over that many bytes
  // (timed: gate/up 14336x4096 x2 21.7-21.9 vs 22.7-22.9 us, the 70B-shape
  // 28672x8192 42.0 vs 43.5 us, the 8B output rows -3%; Q/K/V, o-proj and a
  // single 14336x4096 Q4_0 matrix 0.15-1.5 us slower with them).  The digit
  // variant has its own LDS size, occupancy and grid.
  if constexpr (PkFmt<T>::INTX) {
    const uint64_t rows_pw = (tasks * U + grid * nw - 1) / (grid * nw);
    const uint64_t code_bytes = rows_pw * a.in_dim / PkFmt<T>::EPB * (EPI == EPI_SWIGLU ? 2 : 1);
    const uint64_t lds_ix = pk_digit_lds(T, a.in_dim);
    const bool want = g_digits == 2 || (g_digits == 1 && code_bytes >= 24576);
    if (want && lds_ix + PK_STATIC_LDS <= pk_lds_limit()) {
      auto kix = matvec_packed<T, EPI, NORM, U, LPW, NB, NT, true>;
      const int occ_ix = pk_occupancy(cache_ix, reinterpret_cast<const void*>(kix), NT, (uint32_t)lds_ix, st);
      if (occ_ix < 0) return hipErrorStreamCaptureUnsupported;
      if (occ_ix < 1) return hipErrorInvalidConfiguration;
      note_kernel<T, EPI, NORM, U, LPW, NB, NT, true, false, false>();
      RF_KLAUNCH(kix, dim3((uint32_t)pk_grid(tasks, nw, occ_ix, EPI)), dim3(NT), (uint32_t)lds_ix, st, a);
      return hipGetLastError();
    }
  }
  if constexpr ((T & PK_GGUF) == 0) note_kernel<T, EPI, NORM, U, LPW, NB, NT, false, false, false>();
  RF_KLAUNCH(kern, dim3((uint32_t)grid), dim3(NT), lds, st, a);
  return hipGetLastError();
}

// All-in-flight launches (matvec_packed<..., ALLF>): when a row fits one
// step (LPW = the row's chunks) and the grid gives every wavefront one row,
// the wavefront requests it before the x prologue.  rf_tune_packed_inflight
// switches them off (0) or on (1, default).
static int g_inflight = 1;
void set_packed_inflight(int mode) { g_inflight = mode; }
int packed_inflight() { return g_inflight; }

template <uint32_t T, int EPI, bool NORM, int LPW, int NB>
static hipError_t launch_pk_all_nb(const PkKernelArgs<T>& a, uint32_t lds, uint64_t grid, hipStream_t st) {
  if constexpr ((T & PK_GGUF) == 0) note_kernel<T, EPI, NORM, 1, LPW, NB, 512, false, true, false>();
  RF_KLAUNCH((pk_kernel<T, EPI, NORM, LPW, NB, 512, true>()), dim3((uint32_t)grid), dim3(512), lds, st, a);
  return hipGetLastError();
}

// One row per wavefront: the grid is a wavefront per row when the NB = 1
// instance's occupancy holds that many and the two-step ring would give at
// most 2 rows per wavefront (measured on the 8B shapes, Q8_0, A/B on one box:
// o-proj 4096x4096 7.1 -> 6.6 us; Q/K/V with one row per wavefront in 768
// workgroups 8.73 against 8.44 us for the ring's 3 rows in 256; with 1.5
// rows per wavefront 8.33 against 8.21; the 14336-wide down projection 15.5
// against 13.7 us, its x staged in twice as many workgroups, so neither
// takes this shape; nor do Q8_0 rows of 2048 inputs, two chunks (the d-2048
// model's Q/K/V 4.19 / 4.25 against 4.07 / 4.08 us, decode 2,175 against
// 2,181 tok/s), or of 8192, eight chunks (its down projection: 6.3 against
// 5.9 us)).  *done stays false otherwise.
template <uint32_t T, int EPI, bool NORM, int LPW>
static hipError_t launch_pk_all(const PkKernelArgs<T>& a, uint32_t lds, hipStream_t st, bool* done) {
  *done = false;
  static PkOccCache cache;
  auto k1 = pk_kernel<T, EPI, NORM, LPW, 1, 512, true>();
  const int occ = pk_occupancy(cache, reinterpret_cast<const void*>(k1), 512, lds, st);
  if (occ < 0) return hipErrorStreamCaptureUnsupported;
  if (occ < 1) return hipSuccess;
  const uint64_t nw = 8, cus = (uint64_t)pk_cu_count(), tasks = a.rows_total;
  const uint64_t grid = (tasks + nw - 1) / nw;
  // the ring's grid would give at most 2 rows per wavefront (o-proj); at 3
  // (Q/K/V) the ring's 256 workgroups beat 768 one-row ones
  if (grid > cus * (uint64_t)occ || tasks > 2 * cus * nw) return hipSuccess;
  *done = true;
  return launch_pk_all_nb<T, EPI, NORM, LPW, 1>(a, lds, grid, st);
}

// The single-step launch above with x merged from attention chunk records
// (matvec_packed<..., MRG>): Q8_0 rows of 2 or 4 chunks, Q4_0 / Q4_K / Q6_K rows of 1 or 2,
// with the MRG kernel's own occupancy and LDS (x, its unit sums, then the
// records' factors and the heads' 1 / L).
// hipErrorNotSupported when the shape does not take it;
// with launch false it only says so.
static bool pk_merge_shape(uint32_t t, uint64_t in_dim, uint32_t nsplit, uint32_t qh, uint32_t hd, uint32_t* lds) {
  const PkPlan p = plan_packed(t, in_dim);
  if (!p.ok || !g_inflight) return false;
  if (t == T_Q8_0 || t == T_Q4_0) {
    if (g_digits == 2) return false;  // digit planes everywhere: no float-x launch
  }
  const uint64_t nchunk = pk_nchunk(t, in_dim);
  if (!((t == T_Q8_0 && (nchunk == 2 || nchunk == 4)) || ((t == T_Q4_0 || t == T_Q4_K || t == T_Q6_K) && nchunk <= 2)))
    return false;
  if (hd < 16 || (hd & (hd - 1)) != 0 || (uint64_t)qh * hd != in_dim) return false;
  if (nsplit < 1 || nsplit > 8 || qh > 64) return false;  // 8 lanes per head's chunk records
  if (2 * nchunk * 64 * pk_epb(t) > 512) return false;  // two threads per unit of 16 elements
  const uint64_t l = p.lds_bytes + (uint64_t)nsplit * qh * 4 + (uint64_t)qh * 4;  // factors, 1 / L
  if (l + PK_STATIC_LDS > pk_lds_limit()) return false;
  *lds = (uint32_t)l;
  return true;
}

template <uint32_t T, int LPW>
static hipError_t launch_pk_merge(const PkArgs& a, uint32_t lds, bool launch, hipStream_t st) {
  static PkOccCache cache;
  auto k = matvec_packed<T, EPI_RESIDUAL, false, 1, LPW, 1, 512, false, true, true>;
  const int occ = pk_occupancy(cache, reinterpret_cast<const void*>(k), 512, lds, st);
  if (occ < 0) return hipErrorStreamCaptureUnsupported;
  const uint64_t nw = 8, cus = (uint64_t)pk_cu_count(), tasks = a.rows_total;
  const uint64_t grid = (tasks + nw - 1) / nw;
  if (occ < 1 || grid > cus * (uint64_t)occ || tasks > 2 * cus * nw) return hipErrorNotSupported;
  if (!launch) return hipSuccess;
  note_kernel<T, EPI_RESIDUAL, false, 1, LPW, 1, 512, false, true, true>();
  RF_KLAUNCH(k, dim3((uint32_t)grid), dim3(512), lds, st, a);
  return hipGetLastError();
}

// LPW = the row's chunks (one step per row): Q8_0 rows of 2048 or 4096
// inputs, Q4_0 / Q4_K / Q6_K rows of up to 4096 (Q6_K: 110 VGPRs; an
// all-Q6_K 8B model decodes at 534 against 517 tok/s with the merge kernel).
static hipError_t launch_pk_merge_t(uint32_t t, const PkArgs& a, uint32_t lds, bool launch, hipStream_t st) {
  const uint64_t nchunk = pk_nchunk(t, a.in_dim);
  switch (t) {
    case T_Q8_0:
      return nchunk == 4 ? launch_pk_merge<T_Q8_0, 4>(a, lds, launch, st) : launch_pk_merge<T_Q8_0, 2>(a, lds, launch, st);
    case T_Q4_0:
      return nchunk == 2 ? launch_pk_merge<T_Q4_0, 2>(a, lds, launch, st) : launch_pk_merge<T_Q4_0, 1>(a, lds, launch, st);
    case T_Q4_K:
      return nchunk == 2 ? launch_pk_merge<T_Q4_K, 2>(a, lds, launch, st) : launch_pk_merge<T_Q4_K, 1>(a, lds, launch, st);
    case T_Q6_K:
      return nchunk == 2 ? launch_pk_merge<T_Q6_K, 2>(a, lds, launch, st) : launch_pk_merge<T_Q6_K, 1>(a, lds, launch, st);
    default: return hipErrorNotSupported;
  }
}

hipError_t pk_merge_supported(uint32_t t, uint64_t in_dim, uint64_t rows, uint32_t nsplit, uint32_t qh, uint32_t hd,
                              hipStream_t st) {
  uint32_t lds = 0;
  if (rows == 0 || rows > 0xFFFFFFFFull || !pk_merge_shape(t, in_dim, nsplit, qh, hd, &lds))
    return hipErrorNotSupported;
  PkArgs a{};
  a.rows_total = (uint32_t)rows;
  a.in_dim = (uint32_t)in_dim;
  return launch_pk_merge_t(t, a, lds, false, st);
}

// Launch shape, from timing the 8B projections (Q8_0 and Q4_0; 4096 and
// 14336 inputs): one row per wavefront; LPW = chunks per step, up to 4 (2 for
// gate/up, whose step loads two matrices; Q6_K, with three more loads per
// chunk, one less doubling); 1024-thread workgroups when x fills more than
// 40 KB of LDS (two resident workgroups then still give 32 wavefronts per
// CU), else 512 (always 512 for Q6_K gate/up).  Two step buffers: a third
// for the 8B logits rows (97 instead of 77 VGPRs) took them from 85.3 to
// 89.1 us; steps of 8 chunks for the 14336-wide down projection (119
// VGPRs) from 12.5 to 14.1 us.
template <uint32_t T, int EPI, bool NORM>
static hipError_t launch_pk_l(const PkKernelArgs<T>& a, uint32_t lds, hipStream_t st) {
  const uint64_t nchunk = pk_nchunk(T, a.in_dim);
  // All-in-flight shapes: single-matrix float-x launches whose rows are 4
  // chunks (Q8_0) or 2 (Q4_0, Q4_K): in_dim 4096.
  if constexpr (EPI != EPI_SWIGLU && pk_base(T) != T_Q6_K) {
    bool done = false;
    hipError_t e = hipSuccess;
    if (g_inflight && !(PkFmt<T>::INTX && g_digits == 2)) {
      if constexpr (pk_base(T) == T_Q8_0) {
        if (nchunk == 4) e = launch_pk_all<T, EPI, NORM, 4>(a, lds, st, &done);
      } else {
        if (nchunk == 2) e = launch_pk_all<T, EPI, NORM, 2>(a, lds, st, &done);
      }
    }
    if (done || e != hipSuccess) return e;
  }
  uint32_t pref = EPI == EPI_SWIGLU ? 2 : 4;
  if (pk_base(T) == T_Q6_K) pref /= 2;
  uint32_t lpw = 1;
  while (lpw * 2 <= pref && lpw * 2 <= nchunk) lpw *= 2;
  // Q6_K gate/up keeps 512 threads: its two streams of four regions do not
  // fit the 128 VGPRs of a 1024-thread workgroup (that form spilled to
  // scratch), so it is never instantiated.
  constexpr bool WIDE = !(pk_base(T) == T_Q6_K && EPI == EPI_SWIGLU);
  const bool big = WIDE && lds > 40960;
  switch (lpw * 2 + (big ? 1 : 0)) {
    case 2: return launch_pk<T, EPI, NORM, 1, 2, 512>(a, lds, st);
    case 3:
      if constexpr (WIDE) return launch_pk<T, EPI, NORM, 1, 2, 1024>(a, lds, st);
      return hipErrorInvalidValue;
    case 4: return launch_pk<T, EPI, NORM, 2, 2, 512>(a, lds, st);
    case 5:
      if constexpr (WIDE) return launch_pk<T, EPI, NORM, 2, 2, 1024>(a, lds, st);
      return hipErrorInvalidValue;
    case 8:
      if constexpr (pk_base(T) != T_Q6_K && EPI != EPI_SWIGLU) return launch_pk<T, EPI, NORM, 4, 2, 512>(a, lds, st);
      return hipErrorInvalidValue;
    case 9:
      if constexpr (pk_base(T) != T_Q6_K && EPI != EPI_SWIGLU) return launch_pk<T, EPI, NORM, 4, 2, 1024>(a, lds, st);
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

template <uint32_t T>
static hipError_t launch_pk_t(const PkArgs& a, uint32_t lds, int epi, bool norm, hipStream_t st) {
  switch (epi * 2 + (norm ? 1 : 0)) {
    case EPI_STORE * 2: return launch_pk_l<T, EPI_STORE, false>(a, lds, st);
    case EPI_STORE * 2 + 1: return launch_pk_l<T, EPI_STORE, true>(a, lds, st);
    case EPI_RESIDUAL * 2: return launch_pk_l<T, EPI_RESIDUAL, false>(a, lds, st);
    case EPI_RESIDUAL * 2 + 1: return launch_pk_l<T, EPI_RESIDUAL, true>(a, lds, st);
    case EPI_SWIGLU * 2: return launch_pk_l<T, EPI_SWIGLU, false>(a, lds, st);
    case EPI_SWIGLU * 2 + 1: return launch_pk_l<T, EPI_SWIGLU, true>(a, lds, st);
    default: return hipErrorInvalidValue;
  }
}

static bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

hipError_t launch_matvec_packed(uint32_t t, const PkSegDesc* segs, int nseg, const float* x, const float* norm_w,
                                float eps, uint64_t in_dim, int epi, hipStream_t st, int32_t* advance,
                                const PkMerge* mrg) {
  const PkPlan p = plan_packed(t, in_dim);
  if (!p.ok || nseg < 1 || nseg > 3) return hipErrorInvalidValue;
  uint32_t mlds = 0;
  if (mrg) {
    if (epi != EPI_RESIDUAL || norm_w || nseg != 1 || !mrg->ws || !mrg->d_pos ||
        (reinterpret_cast<uintptr_t>(mrg->ws) & 15u) != 0)
      return hipErrorInvalidValue;
    if (!pk_merge_shape(t, in_dim, mrg->nsplit, mrg->qh, mrg->hd, &mlds)) return hipErrorNotSupported;
  }
  if (!al16(x) || (norm_w && !al16(norm_w))) return hipErrorInvalidValue;
  const bool dual = epi == EPI_SWIGLU;
  const int nreg = pk_nreg(t);
  PkArgs a{};
  uint64_t total = 0;
  for (int i = 0; i < nseg; ++i) {
    const PkSegDesc& d = segs[i];
    if (d.row_start + d.rows > d.matrix_rows) return hipErrorInvalidValue;
    if (dual && !d.packed_up) return hipErrorInvalidValue;
    uint64_t off = 0;  // region k starts after regions 0..k-1 of all matrix rows
    for (int k = 0; k < nreg; ++k) {
      const uint64_t rb = pk_row_bytes(t, k, in_dim);
      a.seg[i].reg[k] = static_cast<const uint8_t*>(d.packed) + off + d.row_start * rb;
      if (dual) a.seg[i].reg_up[k] = static_cast<const uint8_t*>(d.packed_up) + off + d.row_start * rb;
      off += d.matrix_rows * rb;
    }
    // 16-byte loads from region 0 (and Q4_K's headers, Q6_K's qh and scales)
    for (int k = 0; k < nreg; ++k) {
      const bool wide = k == 0 || t == T_Q4_K || (t == T_Q6_K && k < 3);
      if (wide && (!al16(a.seg[i].reg[k]) || (dual && !al16(a.seg[i].reg_up[k])))) return hipErrorInvalidValue;
    }
    a.seg[i].y = d.y;
    a.seg[i].res = d.res;
    a.seg[i].row_begin = (uint32_t)total;
    total += d.rows;
  }
  if (total == 0) return hipSuccess;
  if (total > 0xFFFFFFFFull) return hipErrorInvalidValue;
  a.nseg = (uint32_t)nseg;
  a.rows_total = (uint32_t)total;
  a.x = x;
  a.norm_w = norm_w;
  a.eps = eps;
  a.in_dim = (uint32_t)in_dim;
  a.advance = advance;
  if (mrg) {
    a.mws = mrg->ws;
    a.m_pos = mrg->d_pos;
    a.m_nsplit = mrg->nsplit;
    a.m_qh = mrg->qh;
    a.m_hd_log2 = (uint32_t)__builtin_ctz(mrg->hd);
    return launch_pk_merge_t(t, a, mlds, true, st);
  }
  switch (t) {
    case T_Q8_0: return launch_pk_t<T_Q8_0>(a, p.lds_bytes, epi, norm_w != nullptr, st);
    case T_Q4_0: return launch_pk_t<T_Q4_0>(a, p.lds_bytes, epi, norm_w != nullptr, st);
    case T_Q4_K: return launch_pk_t<T_Q4_K>(a, p.lds_bytes, epi, norm_w != nullptr, st);
    case T_Q6_K: return launch_pk_t<T_Q6_K>(a, p.lds_bytes, epi, norm_w != nullptr, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_matvec_gguf(uint32_t t, const void* w, uint64_t rows, const float* x, float* y, uint64_t in_dim,
                              const PkPlan& p, hipStream_t st) {
  if (!p.ok || !al16(x) || rows > 0x7FFFFFFFull) return hipErrorInvalidValue;
  if (rows == 0) return hipSuccess;
  const PkPlainArgs a{static_cast<const uint8_t*>(w), x, y, (uint32_t)rows, (uint32_t)in_dim};
  const bool dword = (reinterpret_cast<uintptr_t>(w) & 3u) == 0 && (in_dim / pk_qk(t)) % 2 == 0;
  switch (t) {
    case T_Q8_0:
      if (dword) return launch_pk_l<T_Q8_0 | PK_GGUF | PK_DWORD, EPI_STORE, false>(a, p.lds_bytes, st);
      return launch_pk_l<T_Q8_0 | PK_GGUF, EPI_STORE, false>(a, p.lds_bytes, st);
    case T_Q4_0:
      if (dword) return launch_pk_l<T_Q4_0 | PK_GGUF | PK_DWORD, EPI_STORE, false>(a, p.lds_bytes, st);
      return launch_pk_l<T_Q4_0 | PK_GGUF, EPI_STORE, false>(a, p.lds_bytes, st);
    case T_Q5_0: return launch_pk_l<T_Q5_0 | PK_GGUF, EPI_STORE, false>(a, p.lds_bytes, st);
    case T_Q4_K: return launch_pk_l<T_Q4_K | PK_GGUF, EPI_STORE, false>(a, p.lds_bytes, st);
    case T_Q5_K: return launch_pk_l<T_Q5_K | PK_GGUF, EPI_STORE, false>(a, p.lds_bytes, st);
    default:
      if (dword) return launch_pk_l<T_Q6_K | PK_GGUF | PK_DWORD, EPI_STORE, false>(a, p.lds_bytes, st);
      return launch_pk_l<T_Q6_K | PK_GGUF, EPI_STORE, false>(a, p.lds_bytes, st);
  }
}

hipError_t launch_pack(uint32_t t, const void* raw, void* packed, uint64_t rows, uint64_t in_dim, hipStream_t st) {
  if (!packed_type(t) || in_dim % pk_qk(t) != 0) return hipErrorInvalidValue;
  const uint64_t n = rows * (in_dim / pk_qk(t));
  if (n == 0) return hipSuccess;
  const uint32_t gb = n / rows == in_dim / pk_qk(t) ? grid_blocks(n, 256) : 0u;
  if (!gb) return hipErrorInvalidValue;
  const dim3 grid(gb);
  const uint8_t* r = static_cast<const uint8_t*>(raw);
  uint8_t* o = static_cast<uint8_t*>(packed);
  switch (t) {
    case T_Q8_0: RF_KLAUNCH(pack_blocks<T_Q8_0>, grid, dim3(256), 0, st, r, o, n); break;
    case T_Q4_0: RF_KLAUNCH(pack_blocks<T_Q4_0>, grid, dim3(256), 0, st, r, o, n); break;
    case T_Q4_K: RF_KLAUNCH(pack_blocks<T_Q4_K>, grid, dim3(256), 0, st, r, o, n); break;
    default: RF_KLAUNCH(pack_blocks<T_Q6_K>, grid, dim3(256), 0, st, r, o, n); break;
  }
  return hipGetLastError();
}

// Loads this file's code object on the current device (HIP defers that to a
// kernel's first use, which may otherwise fall inside a stream capture) and
// caches the device limits the launchers read.
hipError_t load_module_packed() {
  (void)pk_cu_count();
  (void)pk_lds_limit();
  hipFuncAttributes fa;
  return hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(pack_blocks<T_Q8_0>));
}

}  // namespace rf
