// prefill.hip -- the many-token matmul (prefill chunks, tokens > 8) on the
// matrix cores: v_mfma_f32_32x32x16_f16, gfx950.
//
// y[t * ldy + r] = epilogue(sum_k W[r][k] * x[t][k]) for every kind of the
// decode path, at roughly float32 accuracy although the multiplier takes
// half precision operands:
//
//  * Activations.  Token t is scaled by a power of two 2^-e_t so its largest
//    |x| lies in [2^13, 2^14), then each value is split into two halves,
//    x' = hi + lo with hi = f16(x') and lo = f16(x' - hi): 22 significant bits
//    (prefill_prep_kernel).  The scale comes back once, on the finished sum.
//  * Weights enter as the integer codes of the format, which half precision
//    holds exactly: sc * q for Q4_K and Q5_K (at most 63 * 31), the signed
//    code for the 32-value kinds (q - 8, q - 16, the int8 of Q8_0, or q), and
//    sc * (q - 32) for Q6_K split into its even part and its low bit (up to
//    4096 in magnitude, one bit more than half precision carries).  Every
//    product code * hi, code * lo is then exact in the float32 accumulator.
//  * The scale of a weight block multiplies the accumulator once per block
//    (per 256 values for the K-quants, per 32 for the others), and the
//    min terms (dmin * m of the K-quants, m of Q4_1 / Q5_1) are one more MFMA
//    per 256 values against the per-32 means of x (hi and lo in the 16
//    K-slots; a sum of 32 scaled values would overflow a half).
//
// Against the float32 host dot this differs by float32 rounding of the sums.
// The reference's own tensor-core tile (src/molla/nn/gpu.mojo:2665
// planar_nvmma_kernel) rounds the activations and weights to half precision
// and is held to 2e-3 of the peak; this form keeps the 1e-5 gate of its float
// tiles (tests/test_gpu.mojo:255-300).
//
// Work decomposition.  One MFMA is 32 tokens (M) x 32 rows (N) x 16 values
// (K): lane l holds token / row l % 32 and 8 values of half l / 32 of the step
// (which ones: "The order of K" below), and accumulator element j belongs to
// token 8 (j / 4) + 4 (l / 32) + j % 4, row l % 32.  A wave owns RT row tiles x
// TT token tiles; the waves of a block share its tokens, whose activation
// halves come to LDS 64 values at a time (two buffers), while each wave decodes
// its own rows' weight codes straight from global memory, loaded ahead.  K is
// cut between groups of a block's waves and, where the output tiles are too few
// for the chip, across blockIdx.z, with partial sums in the workspace and a
// second kernel adding them in split order (deterministic) before the
// epilogue.  Rows may come from up to three matrices of one kind laid end to
// end (RowSegs: a layer's q|k|v in one launch), and one activation prep
// (prefill_prepare) can serve several launches over the same input.
//
// Replaces device_matmul_into's batched kernels (src/molla/nn/gpu.mojo:1809
// planar_matmul_kernel, :2665 planar_nvmma_kernel; dispatch :3015) for
// tokens above the decode batch; output layout and epilogues as
// gpu.mojo:1005 and :2955-2961.
#include <algorithm>
#include <type_traits>

#include "matvec_rows.h"

namespace mi {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

constexpr int kTileTok = 32;     // tokens of one MFMA tile
constexpr int kStage = 64;       // values of K per LDS stage (4 MFMA steps)
constexpr int kChunk = 256;      // values per min-term MFMA / K-quant superblock
constexpr int kPadTiles = 4;     // token tiles the activation prep pads to (the widest block's)

__device__ __forceinline__ v16f mfma(v8h a, v8h b, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ v8h as_v8h4(v4u u) { return __builtin_bit_cast(v8h, u); }
// 16 bytes from a 2-byte aligned address (Q6_K's 210-byte superblocks), one
// load: the memory path takes any alignment of whole bytes here.
typedef uint32_t v4u_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32_a2 __attribute__((aligned(2)));
__device__ __forceinline__ v4u ld16(const uint8_t* p) { return *(const v4u_a2*)p; }
__device__ __forceinline__ uint32_t ld4u(const uint8_t* p) { return *(const u32_a2*)p; }
__device__ __forceinline__ uint32_t ld2(const uint8_t* p) { return *(const uint16_t*)p; }
__device__ __forceinline__ float f16f(uint32_t bits) { return half_bits_to_float(bits & 0xFFFF); }

typedef _Float16 v2h __attribute__((ext_vector_type(2)));
__device__ __forceinline__ v2h as_v2h(uint32_t u) { return __builtin_bit_cast(v2h, u); }
__device__ __forceinline__ uint32_t as_u32(v2h h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ v2h splat2(float v) { return v2h{(_Float16)v, (_Float16)v}; }

// Codes are made from "magic" halves: 0x64 above a byte u is the half 1024 + u.
// pair(x, m): the fields m of bytes 0 and 2 of x as two such halves (x >> 8:
// of bytes 1 and 3); a field of bits 4..7 gives 1024 + 16 u.
constexpr uint32_t kMagic = 0x64006400u, kLow = 0x000F000Fu, kHigh = 0x00F000F0u;
__device__ __forceinline__ uint32_t pair(uint32_t x, uint32_t m) { return (x & m) | kMagic; }
__device__ __forceinline__ v8h join(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return __builtin_bit_cast(v8h, v4u{a, b, c, d});
}
// The eight byte pairs' halves (1024 + u) * s + o, one rounding of an exact
// small integer.
__device__ __forceinline__ v8h scaled(v4u p, v2h s, v2h o) {
  v4u r;
#pragma unroll
  for (int i = 0; i < 4; i++) r[i] = as_u32(__builtin_elementwise_fma(as_v2h(p[i]), s, o));
  return __builtin_bit_cast(v8h, r);
}
__device__ __forceinline__ v8h offset(v4u p, v2h o) {
  v4u r;
#pragma unroll
  for (int i = 0; i < 4; i++) r[i] = as_u32(as_v2h(p[i]) + o);
  return __builtin_bit_cast(v8h, r);
}

// The 6-bit scales and mins of groups 0..7 from scales[0..11] held in y, z,
// w (quant.mojo:161 _k_scale), four to a dword.
__device__ __forceinline__ void kscales(uint32_t y, uint32_t w, uint32_t& lo, uint32_t& hi) {
  lo = y & 0x3F3F3F3Fu;
  hi = (w & 0x0F0F0F0Fu) | ((y >> 2) & 0x30303030u);
}
__device__ __forceinline__ v8h kmins(uint32_t z, uint32_t w) {
  uint32_t lo, hi;
  kscales(z, w >> 4, lo, hi);
  const v2h o = splat2(-1024.0f);
  const v4u p = {__builtin_amdgcn_perm(0x64646464u, lo, 0x04010400u), __builtin_amdgcn_perm(0x64646464u, lo, 0x04030402u),
                 __builtin_amdgcn_perm(0x64646464u, hi, 0x04010400u), __builtin_amdgcn_perm(0x64646464u, hi, 0x04030402u)};
  return offset(p, o);
}
// scale j of a superblock in both halves; as a sixteenth (0x54 above a byte
// is 64 + u / 16) for codes left in bits 4..7
__device__ __forceinline__ v2h kscale2(uint32_t lo, uint32_t hi, int j, bool sixteenth) {
  const uint32_t b = (uint32_t)(j & 3), sel = 0x04000400u | (b << 16) | b;
  return sixteenth ? as_v2h(__builtin_amdgcn_perm(0x54545454u, j < 4 ? lo : hi, sel)) + splat2(-64.0f)
                   : as_v2h(__builtin_amdgcn_perm(0x64646464u, j < 4 ? lo : hi, sel)) + splat2(-1024.0f);
}

// ---- per-kind weight access ------------------------------------------------
// The order of K.  MFMA step a (0, 1) of a 32-value group takes, in slot i of
// half wave kh, value 16 kh + 8 a + 4 (i / 4) + {0, 2, 1, 3}[i % 4]: a lane's
// values of a group are 16 consecutive ones (one 16-byte load of a stage
// instead of two of 8), and a dword's bytes pair up as (0, 2), (1, 3), which
// one AND-OR turns into two halves.  prefill_prep_kernel lays the activations
// out in the same order.
//
// Raw: what a lane reads of a row for one stage (64 values of K), SLOTS - 1
// stages ahead, in at least LOADS load instructions; Hdr: what it reads once a 256-value chunk (the K-quants'
// scales), a chunk ahead.  codes(raw, hdr, C, s4, kh, b0, b1): step s4 (0..3)
// of stage C of the chunk, b1 only when LIMBS == 2.
// GROUP: values per block scale.  MIN: 0 none, 1 K-quant dmin * m (scaled per
// superblock), 2 m per 32-value block (Q4_1, Q5_1).
struct NoHdr {};

struct KQ4K {
  static constexpr int GROUP = 256, LIMBS = 1, MIN = 1, BLOCK = 144, SLOTS = 4, LOADS = 1;
  struct Raw {
    v4u q;
  };
  struct Hdr {
    v4u h;
  };
  static __device__ __forceinline__ void load(Raw& r, const uint8_t* row, int st, int kh) {
    r.q = *(const v4u*)(row + (int64_t)(st >> 2) * BLOCK + 16 + 32 * (st & 3) + 16 * kh);
  }
  static __device__ __forceinline__ void load_hdr(Hdr& h, const uint8_t* row, int ch, int) {
    h.h = *(const v4u*)(row + (int64_t)ch * BLOCK);
  }
  // group 2 C is the low nibbles of the stage's bytes, 2 C + 1 the high ones
  static __device__ __forceinline__ void codes(const Raw& r, const Hdr& h, int C, int s4, int, v8h& b0, v8h&) {
    uint32_t lo, hi;
    kscales(h.h.y, h.h.w, lo, hi);
    const int up = s4 >> 1;
    const v2h sc = kscale2(lo, hi, 2 * C + up, up);
    const uint32_t m = up ? kHigh : kLow, x = r.q[2 * (s4 & 1)], y = r.q[2 * (s4 & 1) + 1];
    b0 = scaled(v4u{pair(x, m), pair(x >> 8, m), pair(y, m), pair(y >> 8, m)}, sc, sc * splat2(-1024.0f));
  }
  static __device__ __forceinline__ float d(const Raw&, const Hdr& h) { return f16f(h.h.x); }
  static __device__ __forceinline__ float dmin(const Hdr& h) { return f16f(h.h.x >> 16); }
  static __device__ __forceinline__ v8h mins(const Hdr& h) { return kmins(h.h.z, h.h.w); }
};

struct KQ5K {
  static constexpr int GROUP = 256, LIMBS = 1, MIN = 1, BLOCK = 176, SLOTS = 2, LOADS = 1;
  struct Raw {
    v4u q;
  };
  struct Hdr {
    v4u h, qh;
  };
  static __device__ __forceinline__ void load(Raw& r, const uint8_t* row, int st, int kh) {
    r.q = *(const v4u*)(row + (int64_t)(st >> 2) * BLOCK + 48 + 32 * (st & 3) + 16 * kh);
  }
  static __device__ __forceinline__ void load_hdr(Hdr& h, const uint8_t* row, int ch, int kh) {
    h.h = *(const v4u*)(row + (int64_t)ch * BLOCK);
    h.qh = *(const v4u*)(row + (int64_t)ch * BLOCK + 16 + 16 * kh);
  }
  // the fifth bit of value i of group j is bit j of qh byte i: moved to bit 4
  // above a low nibble, bit 8 above a high one left in place
  static __device__ __forceinline__ void codes(const Raw& r, const Hdr& h, int C, int s4, int, v8h& b0, v8h&) {
    uint32_t lo, hi;
    kscales(h.h.y, h.h.w, lo, hi);
    const int up = s4 >> 1, j = 2 * C + up, to = up ? 8 : 4;
    const v2h sc = kscale2(lo, hi, j, up);
    const uint32_t m = up ? kHigh : kLow, mb = up ? 0x01000100u : 0x00100010u;
    v4u p;
#pragma unroll
    for (int w = 0; w < 2; w++) {
      const uint32_t x = r.q[2 * (s4 & 1) + w], f = h.qh[2 * (s4 & 1) + w];
      const uint32_t f0 = to >= j ? f << (to - j) : f >> (j - to);
      const uint32_t f1 = to >= j + 8 ? f << (to - j - 8) : f >> (j + 8 - to);
      p[2 * w] = pair(x, m) | (f0 & mb);
      p[2 * w + 1] = pair(x >> 8, m) | (f1 & mb);
    }
    b0 = scaled(p, sc, sc * splat2(-1024.0f));
  }
  static __device__ __forceinline__ float d(const Raw&, const Hdr& h) { return f16f(h.h.x); }
  static __device__ __forceinline__ float dmin(const Hdr& h) { return f16f(h.h.x >> 16); }
  static __device__ __forceinline__ v8h mins(const Hdr& h) { return kmins(h.h.z, h.h.w); }
};

// Q6_K (quant.mojo:371): stage C of a superblock covers half n = C / 2 and
// quarters 2 (C % 2) + {0, 1}; step s4 is quarter 2 (C % 2) + s4 / 2, a lane's
// values the 16 of scale sc[8 n + 4 (C % 2) + 2 (s4 / 2) + kh].  sc * (q - 32)
// reaches 4096 in magnitude: b0 is its nearest half, b1 the remainder (-1, 0
// or 1), both exact.
struct KQ6K {
  static constexpr int GROUP = 256, LIMBS = 2, MIN = 0, BLOCK = 210, SLOTS = 2, LOADS = 3;
  struct Raw {
    v4u ql[2], qh;
    uint32_t sc, dbits;
  };
  typedef NoHdr Hdr;
  static __device__ __forceinline__ void load(Raw& r, const uint8_t* row, int st, int kh) {
    const uint8_t* b = row + (int64_t)(st >> 2) * BLOCK;
    const int sp = st & 3, n = sp >> 1;
#pragma unroll
    for (int a = 0; a < 2; a++) r.ql[a] = ld16(b + 64 * n + 32 * a + 16 * kh);
    r.qh = ld16(b + 128 + 32 * n + 16 * kh);
    r.sc = ld4u(b + 192 + 8 * n + 4 * (sp & 1));
    r.dbits = ld2(b + 208);
  }
  static __device__ __forceinline__ void load_hdr(Hdr&, const uint8_t*, int, int) {}
  static __device__ __forceinline__ void codes(const Raw& r, const Hdr&, int C, int s4, int kh, v8h& b0, v8h& b1) {
    const int up = C & 1, a = s4 >> 1, kq = 2 * up + a;
    const _Float16 s = (_Float16)(float)(int8_t)(r.sc >> (16 * a + 8 * kh));
    const v2h sc = {s, s};
    v4u p;
#pragma unroll
    for (int w = 0; w < 2; w++) {
      const uint32_t x = r.ql[a][2 * (s4 & 1) + w] >> (4 * up);
      // bits 2 kq, 2 kq + 1 of the byte to bits 4, 5
      const uint32_t f = r.qh[2 * (s4 & 1) + w], f0 = kq <= 2 ? f << (4 - 2 * kq) : f >> (2 * kq - 4);
      const uint32_t u = (x & 0x0F0F0F0Fu) | (f0 & 0x30303030u);
      p[2 * w] = __builtin_amdgcn_perm(0x64646464u, u, 0x04020400u);
      p[2 * w + 1] = __builtin_amdgcn_perm(0x64646464u, u, 0x04030401u);
    }
    v4u c0, c1;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const v2h q = as_v2h(p[i]) + splat2(-1056.0f);  // q - 32, exact
      const v2h v = q * sc;
      c0[i] = as_u32(v);
      c1[i] = as_u32(__builtin_elementwise_fma(q, sc, -v));
    }
    b0 = __builtin_bit_cast(v8h, c0);
    b1 = __builtin_bit_cast(v8h, c1);
  }
  static __device__ __forceinline__ float d(const Raw& r, const Hdr&) { return f16f(r.dbits); }
  static __device__ __forceinline__ float dmin(const Hdr&) { return 0.0f; }
  static __device__ __forceinline__ v8h mins(const Hdr&) { return v8h{}; }
};

// The 32-value kinds: a stage is two blocks; step s4 is step s4 % 2 of block
// s4 / 2.  A nibble block's values 0..15 are its low nibbles and 16..31 its
// high ones, so half wave kh takes nibble kh of every byte.
template <int KIND>
struct KB32 {
  static constexpr int GROUP = 32, LIMBS = 1, SLOTS = 2, LOADS = 2;
  static constexpr int MIN = (KIND == MI_Q4_1 || KIND == MI_Q5_1) ? 2 : 0;
  static constexpr int BLOCK = KIND == MI_Q8_0 ? 34 : KIND == MI_Q4_0 ? 18 : KIND == MI_Q4_1 ? 20
                               : KIND == MI_Q5_0 ? 22 : 24;
  // u of the magic halves is the unsigned code; the signed one is u - BIAS
  static constexpr float BIAS = KIND == MI_Q8_0 ? 128.0f : KIND == MI_Q4_0 ? 8.0f : KIND == MI_Q5_0 ? 16.0f : 0.0f;
  static constexpr bool FIVE = KIND == MI_Q5_0 || KIND == MI_Q5_1;
  // A stage is two blocks, for the kinds of 34, 18 and 22 bytes a whole number
  // of dwords: they are read from its start, so that on 4-byte aligned weights
  // every load is aligned, and the first block's codes, two bytes off, are
  // moved into place.  (The loads take 2-byte alignment too.  Read at the
  // codes themselves, half of them two bytes off, a tile of Q4_0 4096x14336
  // that held 4 tokens took 39 us against 27; calls of up to 8 tokens take the
  // kernels of matvec_tile_b32.hip.)
  static constexpr int WORDS = KIND == MI_Q4_0 ? 9 : KIND == MI_Q5_0 ? 11 : KIND == MI_Q8_0 ? 11 : 8 + 2 * (BLOCK - 16) / 4;
  typedef uint32_t v2u_a2 __attribute__((ext_vector_type(2), aligned(2)));
  struct Raw {
    uint32_t w[WORDS];
  };
  typedef NoHdr Hdr;
  static __device__ __forceinline__ void put4(uint32_t* w, const uint8_t* p) {
    const v4u v = *(const v4u_a2*)p;
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = v[i];
  }
  static __device__ __forceinline__ void load(Raw& r, const uint8_t* row, int st, int kh) {
    const uint8_t* b = row + (int64_t)st * (2 * BLOCK);
    if constexpr (KIND == MI_Q4_0) {  // d0 q0 | q0 d1 | q1
      put4(r.w, b);
      r.w[4] = ld4u(b + 16);
      put4(r.w + 5, b + 20);
    } else if constexpr (KIND == MI_Q5_0) {  // d0 h0 q0 d1 | h1 q1
      put4(r.w, b);
      put4(r.w + 4, b + 16);
      const v2u_a2 v = *(const v2u_a2*)(b + 32);
      r.w[8] = v.x, r.w[9] = v.y;
      r.w[10] = ld4u(b + 40);
    } else if constexpr (KIND == MI_Q8_0) {  // half wave kh's 16 bytes of each block, and the two scales
      put4(r.w, b + 16 * kh);
      r.w[4] = ld4u(b + 16 + 16 * kh);
      put4(r.w + 5, b + 36 + 16 * kh);
      r.w[9] = ld4u(b);
      r.w[10] = ld4u(b + 32);
    } else {  // each block: d m [h] q, all aligned
#pragma unroll
      for (int bb = 0; bb < 2; bb++) {
        uint32_t* w = r.w + bb * (WORDS / 2);
        w[0] = *(const uint32_t*)(b + bb * BLOCK);
        if constexpr (FIVE) w[1] = *(const uint32_t*)(b + bb * BLOCK + 4);
        put4(w + WORDS / 2 - 4, b + bb * BLOCK + BLOCK - 16);
      }
    }
  }
  static __device__ __forceinline__ void load_hdr(Hdr&, const uint8_t*, int, int) {}
  static __device__ __forceinline__ uint32_t off2(const Raw& r, int i) {  // the dword two bytes into w[i]
    return __builtin_amdgcn_alignbyte(r.w[i + 1], r.w[i], 2);
  }
  // dword i of block bb's codes
  static __device__ __forceinline__ uint32_t code(const Raw& r, int bb, int i) {
    if constexpr (KIND == MI_Q4_0 || KIND == MI_Q8_0) return bb ? r.w[5 + i] : off2(r, i);
    else if constexpr (KIND == MI_Q5_0) return bb ? r.w[7 + i] : off2(r, 1 + i);
    else return r.w[bb * (WORDS / 2) + WORDS / 2 - 4 + i];
  }
  static __device__ __forceinline__ uint32_t fifth(const Raw& r, int bb) {
    return KIND == MI_Q5_0 ? (bb ? r.w[6] : off2(r, 0)) : r.w[bb * (WORDS / 2) + 1];
  }
  static __device__ __forceinline__ void codes(const Raw& r, const Hdr&, int, int s4, int kh, v8h& b0, v8h&) {
    const int bb = s4 >> 1, a = s4 & 1;
    v4u p;
#pragma unroll
    for (int w = 0; w < 2; w++) {
      uint32_t x = code(r, bb, 2 * a + w);
      if constexpr (KIND == MI_Q8_0) {
        x ^= 0x80808080u;  // int8 + 128
        p[2 * w] = __builtin_amdgcn_perm(0x64646464u, x, 0x04020400u);
        p[2 * w + 1] = __builtin_amdgcn_perm(0x64646464u, x, 0x04030401u);
      } else {
        x >>= 4 * kh;
        p[2 * w] = pair(x, kLow);
        p[2 * w + 1] = pair(x >> 8, kLow);
        if constexpr (FIVE) {
          // bits 0, 2 (1, 3) of the dword's four to bits 4 and 20
          const uint32_t f = (fifth(r, bb) >> (16 * kh)) >> (8 * a + 4 * w);
          p[2 * w] |= ((f & 5u) * 0x40010u) & 0x00100010u;
          p[2 * w + 1] |= (((f >> 1) & 5u) * 0x40010u) & 0x00100010u;
        }
      }
    }
    b0 = offset(p, splat2(-1024.0f - BIAS));
  }
  static __device__ __forceinline__ float d(const Raw& r, int bb) {
    if constexpr (KIND == MI_Q4_0) return f16f(bb ? r.w[4] >> 16 : r.w[0]);
    else if constexpr (KIND == MI_Q5_0) return f16f(bb ? r.w[5] >> 16 : r.w[0]);
    else if constexpr (KIND == MI_Q8_0) return f16f(bb ? r.w[10] >> 16 : r.w[9]);
    else return f16f(r.w[bb * (WORDS / 2)]);
  }
  static __device__ __forceinline__ uint32_t mbits(const Raw& r, int bb) { return r.w[bb * (WORDS / 2)] >> 16; }
  // (the K-quants' end of a superblock, which never runs for these)
  static __device__ __forceinline__ float d(const Raw&, const Hdr&) { return 0.0f; }
  static __device__ __forceinline__ float dmin(const Hdr&) { return 0.0f; }
  static __device__ __forceinline__ v8h mins(const Hdr&) { return v8h{}; }
};

template <int KIND> struct KindOf;
template <> struct KindOf<MI_Q4_K> { using T = KQ4K; };
template <> struct KindOf<MI_Q5_K> { using T = KQ5K; };
template <> struct KindOf<MI_Q6_K> { using T = KQ6K; };
template <> struct KindOf<MI_Q8_0> { using T = KB32<MI_Q8_0>; };
template <> struct KindOf<MI_Q4_0> { using T = KB32<MI_Q4_0>; };
template <> struct KindOf<MI_Q4_1> { using T = KB32<MI_Q4_1>; };
template <> struct KindOf<MI_Q5_0> { using T = KB32<MI_Q5_0>; };
template <> struct KindOf<MI_Q5_1> { using T = KB32<MI_Q5_1>; };

// ---- activations -----------------------------------------------------------
// Layout (ttp token tiles of 32, ks = cols / 16 steps, nch = ceil(cols/256)):
//   xp: [tile][step][limb][lane][8 halves]: lane (kh, m) holds token
//       32 tile + m, its slots of the step (the order of K above); limb 0 = hi,
//       1 = lo.
//   xm: [tile][chunk][lane][8 halves]: lane (0, m) holds hi of the means of
//       the chunk's eight 32-value blocks for token 32 tile + m, lane (1, m)
//       their lo (zero past cols).
//   xs: [32 ttp] the power of two each token's sums are multiplied by.
struct Prep {
  int ttp, ks, nch;
  size_t xp, xm, xs, total;
};

__host__ __device__ inline Prep prep_layout(int cols, int tokens) {
  Prep p;
  const int tt = (tokens + kTileTok - 1) / kTileTok;
  p.ttp = (tt + kPadTiles - 1) / kPadTiles * kPadTiles;
  p.ks = cols / 16;
  p.nch = (cols + kChunk - 1) / kChunk;
  p.xp = 0;
  p.xm = p.xp + (size_t)p.ttp * p.ks * 2048;
  p.xs = p.xm + (size_t)p.ttp * p.nch * 1024;
  p.total = (p.xs + (size_t)p.ttp * kTileTok * 4 + 255) & ~(size_t)255;
  return p;
}

__device__ __forceinline__ void split_half(float v, _Float16& hi, _Float16& lo) {
  hi = (_Float16)v;
  lo = (_Float16)(v - (float)hi);
}

// A token's activations, one block a token (256 threads, 8 consecutive values
// a thread and round): its scale, the power of two 2^e with the largest
// |x| * 2^-e in [2^13, 2^14) (e clamped so that the scale stays a normal
// float; 1 for a zero or padding token), xs[t] = 2^e; its halves; and the
// means of its 32-value groups.  A row of up to 16384 values stays in
// registers between the maximum and the split (one launch and one reading of
// x, where two launches were 9.8 us at 256 x 4096).
constexpr int kPrepRounds = 8;
__global__ __launch_bounds__(256) void prefill_prep_kernel(const float* __restrict__ x, int cols, int tokens,
                                                           uint8_t* __restrict__ work) {
  const Prep P = prep_layout(cols, tokens);
  const int t = blockIdx.x, tile = t >> 5, m = t & 31;
  const int n8 = cols >> 3;  // runs of 8 values
  const float* row = x + (int64_t)t * cols;
  typedef float v4f __attribute__((ext_vector_type(4)));
  __shared__ float red[4];
  v4f v[kPrepRounds][2];
  float mx = 0.0f;
  if (t < tokens) {
#pragma unroll
    for (int k = 0; k < kPrepRounds; k++) {
      const int i = min((int)threadIdx.x + 256 * k, n8 - 1);  // (a repeated run changes no maximum)
      if (256 * k < n8) {
        v[k][0] = *(const v4f*)(row + 8 * i);
        v[k][1] = *(const v4f*)(row + 8 * i + 4);
      }
    }
#pragma unroll
    for (int k = 0; k < kPrepRounds; k++)
      if (256 * k < n8) {
#pragma unroll
        for (int i = 0; i < 8; i++) mx = fmaxf(mx, fabsf(v[k][i >> 2][i & 3]));
      }
    for (int i = threadIdx.x + 256 * kPrepRounds; i < n8; i += 256) {
      const v4f a = *(const v4f*)(row + 8 * i), b = *(const v4f*)(row + 8 * i + 4);
#pragma unroll
      for (int e = 0; e < 4; e++) mx = fmaxf(mx, fmaxf(fabsf(a[e]), fabsf(b[e])));
    }
    mx = lanes::reduce<64>(mx, lanes::Max{});
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  }
  const int e = mx > 0.0f ? min(max(ilogbf(mx) - 13, -100), 100) : 0;
  if (threadIdx.x == 0) ((float*)(work + P.xs))[t] = ldexpf(1.0f, e);
  uint8_t* xp = work + P.xp + (size_t)tile * P.ks * 2048 + 16 * m;
  _Float16* xm = (_Float16*)(work + P.xm) + (size_t)tile * P.nch * 512 + 8 * m;
  auto put = [&](int i, v4f a, v4f b) __attribute__((always_inline)) {
    // run i: values 8 i .. +8, half wave (i >> 1) & 1 of step 2 (i >> 2) + (i & 1)
    v8h hi, lo;
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      constexpr int order[4] = {0, 2, 1, 3};  // the order of K (above)
      const int c = order[k & 3];
      const float f = ldexpf(k < 4 ? a[c] : b[c], -e);
      _Float16 h, l;
      split_half(f, h, l);
      hi[k] = h;
      lo[k] = l;
      sum += f;
    }
    uint8_t* dst = xp + (size_t)(2 * (i >> 2) + (i & 1)) * 2048 + 512 * ((i >> 1) & 1);
    *(v8h*)dst = hi;
    *(v8h*)(dst + 1024) = lo;
    // the mean of the group's 32 values (a mean, since 32 values of up to
    // 2^14 overflow a half): four neighbouring lanes
    sum = lanes::reduce<4>(sum, lanes::Add{}) * (1.0f / 32.0f);
    _Float16 h, l;
    split_half(sum, h, l);
    const int g = i >> 2;
    if ((i & 3) == 0) {
      xm[(size_t)(g >> 3) * 512 + (g & 7)] = h;
      xm[(size_t)(g >> 3) * 512 + 256 + (g & 7)] = l;
    }
  };
  // (n8 is a multiple of 8: a group's four lanes go together)
#pragma unroll
  for (int k = 0; k < kPrepRounds; k++) {
    const int i = threadIdx.x + 256 * k;
    if (i < n8) put(i, t < tokens ? v[k][0] : v4f{}, t < tokens ? v[k][1] : v4f{});
  }
  for (int i = threadIdx.x + 256 * kPrepRounds; i < n8; i += 256)
    put(i, t < tokens ? *(const v4f*)(row + 8 * i) : v4f{}, t < tokens ? *(const v4f*)(row + 8 * i + 4) : v4f{});
  // groups past cols in the last chunk
  for (int g = (cols >> 5) + threadIdx.x; g < 8 * P.nch; g += 256) {
    xm[(size_t)(g >> 3) * 512 + (g & 7)] = (_Float16)0.0f;
    xm[(size_t)(g >> 3) * 512 + 256 + (g & 7)] = (_Float16)0.0f;
  }
}

// ---- the matmul ------------------------------------------------------------
// RT x TT tiles (of 32 rows, 32 tokens) a wave, WR waves over rows, KS groups
// of WR waves over K: group g takes every KS-th 256-value chunk of the block's
// share, and the groups' sums meet in LDS at the end (no partial sums in
// memory, where a second launch added them in 10 us at 14336 x 256).
// What bounds it (14336x4096 Q4_K, 256 tokens: 91 -> 71 us; a call, with the
// activations' launch and no partial sums, 105 -> 79 us): 1056 products of 32
// cycles a wave, two waves a SIMD, are 32 us at the 2.1 GHz it runs at; half of
// the products taken out it takes 59 us, the transfer 65, both 53, the decode
// none: the rest is the LDS reads' latency and the barrier of every stage, with
// two waves a SIMD to hide them.
template <int KIND, int RT, int TT, int WR, int KS>
__global__ __launch_bounds__(WR * KS * 64, (WR * KS + 3) / 4) void prefill_kernel(
    const RowSegs sg, int cols, int tokens, const uint8_t* __restrict__ work, int chunks_per_split,
    float* __restrict__ y, int64_t ldy, int epi, const float* __restrict__ aux, float* __restrict__ part) {
  using K = typename KindOf<KIND>::T;
  constexpr int S = K::SLOTS;
  constexpr int kStageBytes = TT * 4 * 2 * 1024;  // one LDS buffer: TT tiles x 4 steps x 2 halves
  constexpr int kBlockRows = WR * RT * 32;
  constexpr int kX = KS * 2 * kStageBytes;
  static_assert(kX <= 65536, "the transfer's LDS address is 16 bits");
  constexpr int kSum = TT * 32 * kBlockRows * 4;
  __shared__ __attribute__((aligned(16))) uint8_t lds[kX > kSum ? kX : kSum];
  const Prep P = prep_layout(cols, tokens);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave / WR, wr = wave % WR;
  const int n = lane & 31, kh = lane >> 5;
  const int tile0 = blockIdx.y * TT;
  const int nst = cols / kStage;
  const int ch0 = blockIdx.z * chunks_per_split, ch1 = min(ch0 + chunks_per_split, P.nch);
  const int rounds = (ch1 - ch0 + KS - 1) / KS;
  const int rows = sg.end[sg.nseg - 1];
  const int row_base = (blockIdx.x * WR + wr) * (RT * 32);
  const uint8_t* wrow[RT];
#pragma unroll
  for (int rt = 0; rt < RT; rt++) wrow[rt] = rows::seg_row(sg, min(row_base + rt * 32 + n, rows - 1));
  uint8_t(*xl)[kStageBytes] = (uint8_t(*)[kStageBytes])(lds + kg * 2 * kStageBytes);

  // The group's activation stage goes to LDS by the direct path (no registers:
  // there are none to spare), 1 KB a wave and instruction.  The instruction is
  // written out because the compiler orders every LDS read behind the builtin's
  // transfer, also the reads of the other buffer, which wait out a memory
  // latency in every stage; the wait that belongs to it is wait_x, ahead of
  // the barrier after which the buffer is read.
  constexpr int kPieces = kStageBytes / 1024 / WR;
  static_assert(kPieces * 1024 * WR == kStageBytes && (kStageBytes / 1024) % WR == 0, "stage copy");
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds + kg * 2 * kStageBytes;
  const uint32_t lane16 = lane * 16;
  // Stage C of round r is stage C of the group's r-th chunk; one past the
  // share repeats its last stage (in bounds) and counts with factor zero.
  auto stage_of = [&](int r, int C) __attribute__((always_inline)) {
    return min(4 * min(ch0 + r * KS + kg, ch1 - 1) + C, nst - 1);
  };
  auto load_x = [&](int st, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < kPieces; q++) {
      const int kb = wr + q * WR;  // the stage's kb-th KB: tile kb / 8
      const uint8_t* src = work + P.xp + ((size_t)(tile0 + (kb >> 3)) * P.ks + 4 * st) * 2048 + (kb & 7) * 1024;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                   :
                   : "s"(lds0 + buf * kStageBytes + kb * 1024), "v"(lane16), "s"(src)
                   : "memory");  // (m0 is a reserved register: naming it is only warned of)
    }
  };
  // Loads complete in order: with at most N younger ones in flight, the
  // transfer has landed.  N counts the loads issued after it, or fewer
  // (check_waits.py looks the compiled code over for it in every build, and that
  // nothing else uses m0).
  auto wait_x = [&](auto nn) __attribute__((always_inline)) {
    constexpr int N = decltype(nn)::value;
    static_assert(N < 16, "one field of s_waitcnt's encoding");
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
  };

  constexpr int kAhead = 2;  // steps whose activations are on the way from LDS
  constexpr int kFill = 5;   // VALU instructions between two products
  typename K::Raw raw[S][RT];
  typename K::Hdr hdr[RT], hdr_next[RT];
  v16f tot[RT][TT], acc[RT][TT];
  const v16f zero = {};
#pragma unroll
  for (int rt = 0; rt < RT; rt++)
#pragma unroll
    for (int tt = 0; tt < TT; tt++) tot[rt][tt] = zero;
  v4u am[TT];  // min-term A fragments of the chunk
  uint32_t mrec[RT][4];

  auto stage = [&](auto cc, int r) __attribute__((always_inline)) {
    constexpr int C = decltype(cc)::value;
    // all ones while the stage is in the share, else zero: a mask on the scales
    // (and opaque), since a select here became a branch around whole stages
    // and thousands of spilled registers
    uint32_t keep = ch0 + r * KS + kg < ch1 && 4 * (ch0 + r * KS + kg) + C < nst ? 0xffffffffu : 0u;
    asm volatile("" : "+v"(keep));
    auto kept = [&](float v) __attribute__((always_inline)) { return __uint_as_float(__float_as_uint(v) & keep); };
    typename K::Raw(&rw)[RT] = raw[C % S];
    load_x(C < 3 ? stage_of(r, C + 1) : stage_of(r + 1, 0), (C + 1) & 1);
    // the slot that the stage before this one emptied: its next stage
    const int next = C + S - 1 < 4 ? stage_of(r, C + S - 1) : stage_of(r + 1, C + S - 5);
#pragma unroll
    for (int rt = 0; rt < RT; rt++) K::load(raw[(C + S - 1) % S][rt], wrow[rt], next, kh);
    if constexpr (K::MIN != 0 && C == 2) {
      const int ch = min(ch0 + r * KS + kg, ch1 - 1);
#pragma unroll
      for (int tt = 0; tt < TT; tt++)
        am[tt] = *(const v4u*)(work + P.xm + (size_t)((tile0 + tt) * P.nch + ch) * 1024 + lane * 16);
    }
    if constexpr (C == 2) {
#pragma unroll
      for (int rt = 0; rt < RT; rt++) K::load_hdr(hdr_next[rt], wrow[rt], min(ch0 + (r + 1) * KS + kg, ch1 - 1), kh);
    }
    // the loads go out here: the scheduler sank them to their first use at the
    // stage's end, a memory latency in every stage
    __builtin_amdgcn_sched_barrier(0);
    // step (s4, tt): the next step's activations are read, and the next s4's
    // codes made, while this one's products run
    auto read_a = [&](int s4, int tt, v4u(&a)[2]) __attribute__((always_inline)) {
      const uint8_t* base = &xl[C & 1][((tt * 4 + s4) * 2) * 1024 + lane * 16];
      a[0] = *(const v4u*)base;
      a[1] = *(const v4u*)(base + 1024);
    };
    v8h b0[2][RT], b1[2][RT];
    v4u a[kAhead + 1][2];
#pragma unroll
    for (int step = 0; step < kAhead; step++) read_a(step / TT, step % TT, a[step]);
#pragma unroll
    for (int rt = 0; rt < RT; rt++) K::codes(rw[rt], hdr[rt], C, 0, kh, b0[0][rt], b1[0][rt]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s4 = 0; s4 < 4; s4++) {
      const bool fresh = K::GROUP == 32 ? !(s4 & 1) : (C == 0 && s4 == 0);
#pragma unroll
      for (int tt = 0; tt < TT; tt++) {
        const int step = s4 * TT + tt, far = step + kAhead;
        if (far < 4 * TT) read_a(far / TT, far % TT, a[far % (kAhead + 1)]);
        const v8h ahi = as_v8h4(a[step % (kAhead + 1)][0]), alo = as_v8h4(a[step % (kAhead + 1)][1]);
#pragma unroll
        for (int rt = 0; rt < RT; rt++) acc[rt][tt] = mfma(ahi, b0[s4 & 1][rt], fresh ? zero : acc[rt][tt]);
        if constexpr (K::LIMBS == 2) {
#pragma unroll
          for (int rt = 0; rt < RT; rt++) acc[rt][tt] = mfma(ahi, b1[s4 & 1][rt], acc[rt][tt]);
        }
#pragma unroll
        for (int rt = 0; rt < RT; rt++) acc[rt][tt] = mfma(alo, b0[s4 & 1][rt], acc[rt][tt]);
        // the next s4's codes, a row tile in each of the steps
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
          if (s4 < 3 && rt * TT / RT == tt)
            K::codes(rw[rt], hdr[rt], C, s4 + 1, kh, b0[(s4 + 1) & 1][rt], b1[(s4 + 1) & 1][rt]);
        // a product, then what the VALU does in its 32 cycles: in a wave's
        // order of issue the codes would otherwise wait for all of the
        // step's products, and the matrix core for the codes
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
        for (int k = 0; k < RT * (1 + K::LIMBS); k++) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, kFill, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (K::GROUP == 32) {
        if (s4 & 1) {  // a 32-value block ends
          const int bb = s4 >> 1;
#pragma unroll
          for (int rt = 0; rt < RT; rt++) {
            const float dv = kept(K::d(rw[rt], bb));
#pragma unroll
            for (int tt = 0; tt < TT; tt++) tot[rt][tt] += dv * acc[rt][tt];
            if constexpr (K::MIN == 2) {
              const int slot = 2 * C + bb;  // block of the chunk
              const uint32_t mb = K::mbits(rw[rt], bb) & keep;
              mrec[rt][slot >> 1] = (slot & 1) ? (mrec[rt][slot >> 1] | (mb << 16)) : mb;
            }
          }
        }
      }
    }
    if constexpr (K::GROUP == 256 && C == 3) {  // a superblock ends
#pragma unroll
      for (int rt = 0; rt < RT; rt++) {
        const float dv = kept(K::d(rw[rt], hdr[rt]));
#pragma unroll
        for (int tt = 0; tt < TT; tt++) tot[rt][tt] += dv * acc[rt][tt];
        if constexpr (K::MIN == 1) {
          const float dm = kept(32.0f * K::dmin(hdr[rt]));
          const v8h bm = K::mins(hdr[rt]);
#pragma unroll
          for (int tt = 0; tt < TT; tt++) tot[rt][tt] -= dm * mfma(as_v8h4(am[tt]), bm, zero);
        }
      }
    }
    if constexpr (K::MIN == 2 && C == 3) {  // a chunk of eight blocks ends
#pragma unroll
      for (int rt = 0; rt < RT; rt++) {
        const v8h bm = as_v8h4(v4u{mrec[rt][0], mrec[rt][1], mrec[rt][2], mrec[rt][3]});
#pragma unroll
        for (int tt = 0; tt < TT; tt++) {
          __builtin_amdgcn_sched_barrier(0);
          tot[rt][tt] += 32.0f * mfma(as_v8h4(am[tt]), bm, zero);
        }
      }
    }
    wait_x(std::integral_constant<int, RT * K::LOADS + (C == 2 ? (K::MIN ? TT : 0) + (K::GROUP == 256 && K::MIN ? RT : 0) : 0)>{});
    if constexpr (C == 3) {
#pragma unroll
      for (int rt = 0; rt < RT; rt++) hdr[rt] = hdr_next[rt];
    }
    __syncthreads();
  };

  load_x(stage_of(0, 0), 0);
#pragma unroll
  for (int rt = 0; rt < RT; rt++) {
    K::load_hdr(hdr[rt], wrow[rt], min(ch0 + kg, ch1 - 1), kh);
#pragma unroll
    for (int q = 0; q < 4; q++) mrec[rt][q] = 0;
  }
#pragma unroll
  for (int c = 0; c < S - 1; c++)
#pragma unroll
    for (int rt = 0; rt < RT; rt++) K::load(raw[c][rt], wrow[rt], stage_of(0, c), kh);
  wait_x(std::integral_constant<int, 0>{});
  __syncthreads();
  for (int r = 0; r < rounds; r++) {
    stage(std::integral_constant<int, 0>{}, r);
    stage(std::integral_constant<int, 1>{}, r);
    stage(std::integral_constant<int, 2>{}, r);
    stage(std::integral_constant<int, 3>{}, r);
  }

  // The K groups' sums meet in LDS, in group order, and leave it by rows, so
  // that the epilogue's code runs once and not once for each of a lane's 64
  // results (15 us of 84 at 14336 x 4096 x 256).  The loop's last barrier has
  // passed: the activation buffers are free.  Element j of tile (rt, tt) is
  // token 32 tt + 8 (j / 4) + 4 kh + j % 4, row 32 rt + n of the wave's.
  float* sum = (float*)lds + wr * (RT * 32) + n;
#pragma unroll
  for (int g = KS - 1; g >= 0; g--) {
    if (kg == g) {
#pragma unroll
      for (int tt = 0; tt < TT; tt++)
#pragma unroll
        for (int j = 0; j < 16; j++)
#pragma unroll
          for (int rt = 0; rt < RT; rt++) {
            float* at = sum + (32 * tt + 8 * (j >> 2) + 4 * kh + (j & 3)) * kBlockRows + rt * 32;
            *at = g == KS - 1 ? tot[rt][tt][j] : tot[rt][tt][j] + *at;
          }
    }
    __syncthreads();
  }
  const float* xs = (const float*)(work + P.xs);
  const int row0 = blockIdx.x * kBlockRows, t0 = tile0 * 32;
  static_assert(kBlockRows % 64 == 0, "a wave takes one token's rows");
#pragma unroll 4
  for (int tl = wave; tl < TT * 32; tl += WR * KS) {
    const int t = t0 + tl;
    if (t >= tokens) break;
    const float sc = xs[t];
#pragma unroll
    for (int k = 0; k < kBlockRows / 64; k++) {
      const int r = row0 + 64 * k + lane;
      const float v = ((const float*)lds)[tl * kBlockRows + 64 * k + lane] * sc;
      if (r >= rows) continue;
      if (part) part[((size_t)blockIdx.z * tokens + t) * rows + r] = v;
      else mv::epilogue(y, aux, epi, (int64_t)t * ldy + r, r, v);
    }
  }
}

// Adds the splits' partial sums in split order and applies the epilogue.
__global__ __launch_bounds__(256) void prefill_reduce_kernel(const float* __restrict__ part, int splits, int rows,
                                                             int tokens, float* __restrict__ y, int64_t ldy, int epi,
                                                             const float* __restrict__ aux) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t n = (int64_t)rows * tokens;
  if (i >= n) return;
  float v = part[i];
  for (int z = 1; z < splits; z++) v += part[z * n + i];
  const int t = (int)(i / rows), r = (int)(i - (int64_t)t * rows);
  mv::epilogue(y, aux, epi, (int64_t)t * ldy + r, r, v);
}

// How a block is cut: (row tiles, token tiles) of 32 a wave, waves over rows,
// groups over K.
struct Shape {
  int rt, tt, wr, ks;
  int block_rows() const { return wr * rt * 32; }
};
// Each measured against the others (us a call).  Up to 32 tokens (1, 1, 4, 2) /
// (1, 2, 4, 2) / (1, 1, 4, 4): Q4_K 4096x4096 12.7 / 13.8 / 13.5, Q6_K 17.2 / - /
// 22.9, Q8_0 17.7 / 19.1 / 24.6.
// Small matrices want more, smaller blocks.  (1, 2, 4, 2) / (2, 2, 4, 2) by `work`,
// the 256-value chunks of 256 x 64 outputs:
//   896   14336x4096, 64 tokens   Q4_K 35.6 / 37.9  Q8_0 44.5 / 47.9  Q4_0 39.0 / 39.3
//   1232  5632x2048, 400          Q4_K 54.2 / 44.8  Q8_0 59.7 / 61.9  Q4_0 48.8 / 51.2
//   1536  6144x4096, 256          Q4_K 47.3 / 49.5  Q8_0 65.5 / 66.8  Q4_0 60.5 / 56.0
//   1792  14336x4096, 128         Q4_K 47.6 / 51.7  Q8_0 68.5 / 72.3  Q4_0 58.1 / 55.8
//   2064  11008x4096, 192         Q4_K 87.3 / 65.5  Q8_0 107.9 / 105.9  Q4_0 80.5 / 83.2
//   2688  4096x14336, 192         Q4_K 82.1 / 76.9  Q8_0 122.7 / 116.1  Q4_0 103.2 / 88.8
//   3584  14336x4096, 256         Q4_K 89.8 / 77.8  Q8_0 111.5 / 113.9  Q4_0 87.7 / 86.4
// The line is a rough one: the smaller blocks lose where they need a second round
// of the chip (up to 25 %) and for Q4_K and Q8_0 win up to there, to 2048 (11 %).
// Q6_K, three products a step, pays for the larger token tile also where half of
// it is empty: (1, 2, 4, 2) / (2, 2, 4, 2) / (1, 4, 8, 1) 14336x4096 at 96 tokens
// 68 / 73 / 62, at 128 69 / 74 / 68, at 150 124 / 117 / 98, 4096x14336 at 192 121 /
// 120 / 107, at 256 127 / 127 / 114; at 64 48 / 54 / 62.
// (The (2, 2, 4, 2) block of Q5_1 spills 10 registers in its stage and is still the
// faster one at 14336x4096, 256 tokens: 118 / 106.)
Shape shape_for(int kind, int rows, int cols, int tokens) {
  if (tokens <= 32) return Shape{1, 1, 4, 2};
  const int64_t work = (int64_t)((rows + 255) / 256) * ((tokens + 63) / 64) * ((cols + kChunk - 1) / kChunk);
  if (work <= 1536) return Shape{1, 2, 4, 2};
  if (kind == MI_Q6_K && tokens > 64) return Shape{1, 4, 8, 1};
  return Shape{2, 2, 4, 2};
}

template <int KIND>
int launch_kind(hipStream_t s, const RowSegs& sg, int cols, int tokens, const void* work, int splits, int cps,
                float* y, int64_t ldy, int epi, const float* aux, float* part) {
  const int rows = sg.end[sg.nseg - 1];
  const Shape sh = shape_for(KIND, rows, cols, tokens);
  const int tiles = (tokens + kTileTok - 1) / kTileTok;
  const dim3 grid((rows + sh.block_rows() - 1) / sh.block_rows(), (tiles + sh.tt - 1) / sh.tt, splits);
  const dim3 block(sh.wr * sh.ks * 64);
#define MI_PF(R, T, W, G)                                                                                  \
  hipLaunchKernelGGL((prefill_kernel<KIND, R, T, W, G>), grid, block, 0, s, sg, cols, tokens,               \
                     (const uint8_t*)work, cps, y, ldy, epi, aux, splits > 1 ? part : nullptr)
  if (sh.tt == 1) MI_PF(1, 1, 4, 2);
  else if (sh.rt == 1 && sh.tt == 2) MI_PF(1, 2, 4, 2);
  else if constexpr (KIND == MI_Q6_K) {
    if (sh.tt == 4) MI_PF(1, 4, 8, 1);
    else MI_PF(2, 2, 4, 2);
  } else {
    MI_PF(2, 2, 4, 2);
  }
#undef MI_PF
  return hip_check(hipGetLastError(), "prefill launch");
}

// Splits of K over blocks (in whole 256-value chunks): the largest power of
// two whose blocks still fit one round of the chip, one block a compute unit,
// each K group of a block at least one chunk.
int choose_splits(int kind, int rows, int cols, int tokens) {
  const Shape sh = shape_for(kind, rows, cols, tokens);
  const int tiles = (tokens + kTileTok - 1) / kTileTok;
  const int64_t blocks = (int64_t)((rows + sh.block_rows() - 1) / sh.block_rows()) * ((tiles + sh.tt - 1) / sh.tt);
  const int chunks = (cols + kChunk - 1) / kChunk;
  int s = 1;
  const int places = cu_count();
  while (blocks * 2 * s <= places && chunks >= 2 * s * sh.ks) s *= 2;
  return s;
}

}  // namespace

bool prefill_fits(int kind, int32_t cols, int64_t row_bytes, const void* w) {
  if (cols % kStage) return false;
  switch (kind) {
    case MI_Q4_K:
    case MI_Q5_K:
      return cols % 256 == 0 && ((uintptr_t)w & 15) == 0 && row_bytes % 16 == 0;
    case MI_Q6_K:
      return cols % 256 == 0 && ((uintptr_t)w & 1) == 0 && row_bytes % 2 == 0;
    case MI_Q4_1:
      return ((uintptr_t)w & 3) == 0 && row_bytes % 4 == 0;
    case MI_Q5_1:
      return ((uintptr_t)w & 7) == 0 && row_bytes % 8 == 0;
    case MI_Q8_0:
    case MI_Q4_0:
    case MI_Q5_0:
      return ((uintptr_t)w & 1) == 0 && row_bytes % 2 == 0;
  }
  return false;
}

size_t prefill_workspace(int32_t rows, int32_t cols, int32_t tokens) {
  const Prep P = prep_layout(cols, tokens);
  int splits = 1;  // the most any kind takes (shape_for tells two apart)
  for (int k : {MI_Q4_K, MI_Q6_K}) splits = std::max(splits, rows > 0 ? choose_splits(k, rows, cols, tokens) : 1);
  size_t part = splits > 1 ? (size_t)splits * tokens * rows * 4 : 0;
  return P.total + ((part + 255) & ~(size_t)255);
}

size_t prefill_prep_bytes(int32_t cols, int32_t tokens) { return prep_layout(cols, tokens).total; }

int prefill_prepare(hipStream_t s, const float* x, int32_t cols, int32_t tokens, void* work) {
  const Prep P = prep_layout(cols, tokens);
  hipLaunchKernelGGL(prefill_prep_kernel, dim3(P.ttp * kTileTok), dim3(256), 0, s, x, cols, tokens, (uint8_t*)work);
  return hip_check(hipGetLastError(), "prefill activation launch");
}

int launch_prefill_segs(hipStream_t s, int kind, const RowSegs& sg, int32_t cols, int32_t tokens, float* y,
                        int64_t ldy, int32_t epi, const float* aux, void* work, size_t work_bytes) {
  const Prep P = prep_layout(cols, tokens);
  const int rows = sg.end[sg.nseg - 1];
  int splits = choose_splits(kind, rows, cols, tokens);
  const size_t need = (size_t)splits * tokens * rows * 4;
  if (splits > 1 && work_bytes < P.total + need) splits = 1;  // no room for partial sums
  const int cps = (P.nch + splits - 1) / splits;
  splits = (P.nch + cps - 1) / cps;
  float* part = (float*)((uint8_t*)work + P.total);
  int rc;
  switch (kind) {
    case MI_Q4_K: rc = launch_kind<MI_Q4_K>(s, sg, cols, tokens, work, splits, cps, y, ldy, epi, aux, part); break;
    case MI_Q5_K: rc = launch_kind<MI_Q5_K>(s, sg, cols, tokens, work, splits, cps, y, ldy, epi, aux, part); break;
    case MI_Q6_K: rc = launch_kind<MI_Q6_K>(s, sg, cols, tokens, work, splits, cps, y, ldy, epi, aux, part); break;
    case MI_Q8_0: rc = launch_kind<MI_Q8_0>(s, sg, cols, tokens, work, splits, cps, y, ldy, epi, aux, part); break;
    case MI_Q4_0: rc = launch_kind<MI_Q4_0>(s, sg, cols, tokens, work, splits, cps, y, ldy, epi, aux, part); break;
    case MI_Q4_1: rc = launch_kind<MI_Q4_1>(s, sg, cols, tokens, work, splits, cps, y, ldy, epi, aux, part); break;
    case MI_Q5_0: rc = launch_kind<MI_Q5_0>(s, sg, cols, tokens, work, splits, cps, y, ldy, epi, aux, part); break;
    case MI_Q5_1: rc = launch_kind<MI_Q5_1>(s, sg, cols, tokens, work, splits, cps, y, ldy, epi, aux, part); break;
    default: return fail(MI_ERR_KIND, "prefill: ggml type %d has no tile", kind);
  }
  if (rc || splits == 1) return rc;
  const int64_t n = (int64_t)rows * tokens;
  hipLaunchKernelGGL(prefill_reduce_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, part, splits, rows,
                     tokens, y, ldy, epi, aux);
  return hip_check(hipGetLastError(), "prefill reduce launch");
}

int launch_prefill(hipStream_t s, int kind, const void* w, int64_t row_bytes, int32_t rows, int32_t cols,
                   const float* x, int32_t tokens, float* y, int64_t ldy, int32_t epi, const float* aux, void* work,
                   size_t work_bytes) {
  int rc = prefill_prepare(s, x, cols, tokens, work);
  if (rc) return rc;
  return launch_prefill_segs(s, kind, rows::one_matrix(w, row_bytes, rows), cols, tokens, y, ldy, epi, aux, work,
                             work_bytes);
}

}  // namespace mi
