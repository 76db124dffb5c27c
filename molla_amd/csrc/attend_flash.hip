// attend_flash.hip -- a prompt chunk's attention on the matrix cores
// (v_mfma_f32_32x32x16_f16), gfx950: attention.mojo:144 attend for many
// query tokens of one sequence, over an f16 or a q8_0 cache (gpu_ops.mojo:678
// attend_kernel's `form`), GQA, each token over the positions up to its own.
//
// A block holds 128 query rows (128 / group tokens x the group of query heads
// of one key head), 32 to a wave, and walks a run of 64-key slices with a
// running maximum and sum, so a slice's scores and weights never leave the
// registers and only one partial result a block is written.  (One block a
// slice, as the decode kernels do it, wrote 8.9 MB of partials a slice at 256
// tokens x 32 heads: at 4096 keys of context 190 us for the slices and 54 us
// for the merge of a layer's chunk.)
//
//   S^T = K Q^T, keys as rows and queries as columns: a lane's 32 scores of a
//   slice all belong to its own query, so the softmax is in the lane but for
//   one exchange of the two half waves, and the weights are in place as the B
//   operand of the next product.  Queries enter as three halves, each query
//   scaled by a power of two so that its largest value is in [2^14, 2^15): any
//   f32 query, to 2^-39 of its largest value (every bit of values down to 2^-15
//   of it; two halves left 1e-4 of the output at scores of a few hundred).
//   O^T = V^T P^T: values lie by rows in LDS and are read transposed
//   (ds_read_b64_tr_b16); P is lifted by 2^14 and split into two halves, each
//   rounded: to 2^-24 of a weight, as an f32 is (see kLift).  MFMA step u of a
//   32-key tile takes keys 8 (i / 4) + 4 h + i % 4 of its 16 in slot (half wave
//   h, i), the order in which S^T leaves them.
//
// q8_0: keys enter as their integers (exact halves) and each 32-value
// block's factor multiplies that block's part of the score; values enter as
// value * 2^(8 - X) in two halves (7 + 11 bits: exact), X the largest factor's
// exponent so far in that 32-value block; of the four products the one of both
// low halves is left out, at most 2^-24 of the whole.  A key whose factor is
// below 2^(X - 22) (its low half would be subnormal) or not finite is left out of
// the product (its values enter as zeros) and added in float32 at the end, to the
// rows that it is live for: a later token's factor changes nothing of an earlier
// one's result.
//
// MFMA fragments (32x32x16): lane l holds row / column l % 32 and values
// 8 (l / 32) .. +8 of the 16; result element j of lane l is row 8 (j / 4) +
// 4 (l / 32) + j % 4, column l % 32.
//
// What bounds it: 80 MFMA a wave a slice (96 for q8_0; 32 cycles each)
// against ~1300 cycles of softmax on the VALU, two waves a SIMD (the matrix cores
// are busy a third of the time, the VALU half).  256 tokens x 32 heads of 128 (8
// key heads) behind 3840 positions of f16: 244 us (one block a slice, and its
// merge) -> 64 and 9 for the fold; 220 over 1280 positions of q8_0 (the decode
// kernel, a token a block) 494 -> 41.  At D = 128 it spills 5 to 7 registers.
#include <math.h>

#include <algorithm>

#include "mi_internal.h"

namespace mi {
namespace {

typedef _Float16 fh2 __attribute__((ext_vector_type(2)));
typedef _Float16 fh8 __attribute__((ext_vector_type(8)));
typedef short fs4 __attribute__((ext_vector_type(4)));
typedef short fs8 __attribute__((ext_vector_type(8)));
typedef float ff4 __attribute__((ext_vector_type(4)));
typedef float ff16 __attribute__((ext_vector_type(16)));
typedef uint32_t fu4 __attribute__((ext_vector_type(4)));

constexpr int kSlice = 64;    // keys a block takes at a time
constexpr int kRows = 128;    // query rows a block
// P (at most 1) is lifted by 2^14 before it is split into halves, so that the
// low halves of weights down to ~1e-8 are not f16 subnormals, and the sums are
// scaled back.  (A lift in the exponential's argument rounds that to 2^-21, weights
// to 3e-7; after it, it takes 2 us of a layer's 470 at a chunk of 256.)
constexpr float kLift = 16384.0f;
constexpr float kLog2e = 1.44269504088896340736f;

__device__ __forceinline__ ff16 mfma32(fh8 a, fh8 b, ff16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// LDS rows of D halves, in 16-byte pieces.  Piece pc of row r lies at slot
// pc ^ key_swz(r) (keys: 16 lanes read one piece of 16 rows) or pc ^
// val_swz(r) (values: a transposed read takes 4 rows x 32 bytes per 16 lanes),
// so that the lanes served together fall on distinct banks.
template <int D>
__device__ __forceinline__ int key_swz(int r) {
  return D == 128 ? (r & 15) : ((r >> 1) & 7);
}
template <int D>
__device__ __forceinline__ int val_swz(int r) {
  return (D == 128 ? 4 * (r & 3) : 4 * ((r >> 1) & 1)) | ((r >> 2) & 3);
}

struct IMax {
  __device__ __forceinline__ int operator()(int a, int b) const { return max(a, b); }
};

__device__ __forceinline__ float other_max(float v) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
__device__ __forceinline__ float other_sum(float v) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}

// four signed bytes as halves: 0x64 above byte + 128 is 1152 + byte
__device__ __forceinline__ void int8_halves(uint32_t w, fh2& a, fh2& b) {
  const fh2 off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
  w ^= 0x80808080u;
  a = __builtin_bit_cast(fh2, __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u)) + off;
  b = __builtin_bit_cast(fh2, __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u)) + off;
}

// The grid is (splits, kv_heads, token tiles).  Block x takes the x-th share
// of the slices that the tile's farthest token reaches (a device value: the
// host knows only the context), and writes each row's unnormalised sum with
// (maximum, sum) in base 2 to part_acc / part_ml, slot (token, head, split);
// with one split, the finished row to out.
template <int D, bool Q8, bool PAGED>
__global__ __launch_bounds__(256, 2) void attend_flash_kernel(
    const float* __restrict__ q, int64_t q_stride, const __half* __restrict__ kc, const __half* __restrict__ vc,
    int row_halves, int heads, int kv_heads, int group, float scale, const int32_t* __restrict__ pos, int tokens,
    const int32_t* __restrict__ kv_index, float* __restrict__ part_acc, float* __restrict__ part_ml,
    float* __restrict__ out) {
  constexpr int PIECES = D / 8, NT = D / 32;
  constexpr int VB = Q8 ? 1 : 2;  // value buffers (q8_0 values take two halves: 32 KB at D = 128)
  constexpr int VH = Q8 ? 2 : 1;  // halves a value
  __shared__ __align__(16) _Float16 ks[2][kSlice * D];
  __shared__ __align__(16) _Float16 vs[VB * VH][kSlice * D];
  __shared__ __align__(16) float kf[Q8 ? 2 : 1][Q8 ? NT : 1][kSlice];  // q8_0 key factors
  __shared__ int vexp[Q8 ? 4 : 1];                                     // X of each wave's dims
  __shared__ int left_out;                                             // q8_0: some key's values were
  __shared__ int cmax[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int split = blockIdx.x, splits = gridDim.x, kvh = blockIdx.y, t0 = blockIdx.z * (kRows / group);

  // this lane's query: row r = token t0 + r / group, head r % group
  const int r = 32 * wave + n, t = t0 + r / group, head = kvh * group + r % group;
  const bool live_row = t < tokens;
  const int cnt = live_row ? pos[t] + 1 : 0;
  const int wave_max = lanes::reduce<64>(cnt, IMax{});
  const int wave_min = -lanes::reduce<64>(live_row ? -cnt : -0x7fffffff, IMax{});
  if (lane == 0) cmax[wave] = wave_max;
  if (Q8 && tid == 0) left_out = 0;
  __syncthreads();
  const int count = __builtin_amdgcn_readfirstlane(max(max(cmax[0], cmax[1]), max(cmax[2], cmax[3])));
  const int slices = (count + kSlice - 1) / kSlice, per = (slices + splits - 1) / splits;
  const int s0 = split * per, s1 = min(s0 + per, slices);

  if (s0 >= s1) {  // (uniform; only with several splits) no keys: no part in the fold
    if (live_row && h == 0) *(float2*)(part_ml + (((int64_t)t * heads + head) * splits + split) * 2) = make_float2(0.0f, 0.0f);
    return;
  }

  const float* qr = q + (int64_t)min(t, tokens - 1) * q_stride + (int64_t)head * D + 8 * h;
  ff4 qraw[D / 16][2];
#pragma unroll
  for (int st = 0; st < D / 16; st++) {
    qraw[st][0] = *(const ff4*)(qr + 16 * st);
    qraw[st][1] = *(const ff4*)(qr + 16 * st + 4);
  }

  // Staging.  f16: a thread copies pieces tid + 256 j of the slice's rows.
  // q8_0: a thread takes D / 4 values of key `lane` (whole 16-byte words, in
  // one 32-value block).  Keys past the end repeat the last one (masked).
  constexpr int PER = Q8 ? D / 64 : kSlice * PIECES / 256;  // 16-byte words of K (and of V)
  fu4 kr[PER], vr[PER];
  uint16_t kfr = 0, vfr = 0;  // the factor's bits (converted when stored: a use here would wait for the load)
  uint64_t dead = 0;  // q8_0: the loaded slice's keys that no row reaches
  const int kvw = kv_heads * D;
  auto cell_of = [&](int sl, int key) __attribute__((always_inline)) {
    const int j = min(sl * kSlice + key, count - 1);
    return PAGED ? kv_index[j] : j;  // (negative: not held)
  };
  auto row_of = [&](int cell) __attribute__((always_inline)) { return (int64_t)max(cell, 0) * row_halves; };
  auto load = [&](const __half* __restrict__ c, int sl, fu4 (&w)[PER], uint16_t& f) __attribute__((always_inline)) {
    if constexpr (Q8) {
      const int cell = cell_of(sl, lane);
      const __half* rowp = c + row_of(cell);
      const int8_t* b = (const int8_t*)rowp + kvh * D + wave * (D / 4);
#pragma unroll
      for (int j = 0; j < PER; j++) w[j] = *(const fu4*)(b + 16 * j);
      f = ((const uint16_t*)rowp)[(kvw >> 1) + ((kvh * D + wave * (D / 4)) >> 5)];
      dead = __ballot(sl * kSlice + lane >= count || (PAGED && cell < 0));
    } else {
#pragma unroll
      for (int j = 0; j < PER; j++) {
        const int i = tid + 256 * j;
        w[j] = *(const fu4*)(c + row_of(cell_of(sl, i / PIECES)) + kvh * D + 8 * (i % PIECES));
      }
    }
  };
  auto store_k = [&](int buf) __attribute__((always_inline)) {
    if constexpr (Q8) {
#pragma unroll
      for (int j = 0; j < PER; j++) {
        fh8 a[2];
#pragma unroll
        for (int w = 0; w < 4; w++) {
          fh2 lo, hi;
          int8_halves(kr[j][w], lo, hi);
          a[w >> 1][4 * (w & 1)] = lo[0];
          a[w >> 1][4 * (w & 1) + 1] = lo[1];
          a[w >> 1][4 * (w & 1) + 2] = hi[0];
          a[w >> 1][4 * (w & 1) + 3] = hi[1];
        }
        const int pc = wave * (D / 32) + 2 * j;
        *(fh8*)(ks[buf] + lane * D + 8 * (pc ^ key_swz<D>(lane))) = a[0];
        *(fh8*)(ks[buf] + lane * D + 8 * ((pc + 1) ^ key_swz<D>(lane))) = a[1];
      }
      // (at D = 64 two waves share a block and write the same factors)
      kf[buf][wave * (D / 4) / 32][lane] = half_bits_to_float(kfr);
    } else {
#pragma unroll
      for (int j = 0; j < PER; j++) {
        const int i = tid + 256 * j, row = i / PIECES, pc = i % PIECES;
        *(fu4*)(ks[buf] + row * D + 8 * (pc ^ key_swz<D>(row))) = kr[j];
      }
    }
  };
  // q8_0: X with the slice's factors f (lane: key), and whether this lane's key
  // stays out of the product: a half's factor is 11 bits, and down to 2^(X - 22)
  // its products' low halves end at 2^-24
  auto track = [&](float f, int& x) __attribute__((always_inline)) {
    const float af = fabsf(f), fm = lanes::reduce<64>(af < INFINITY ? af : 0.0f, lanes::Max{});
    if (fm > 0.0f) x = max(x, __builtin_amdgcn_frexp_expf(fm));
    x = __builtin_amdgcn_readfirstlane(x);
    return !(af < INFINITY) || (af > 0.0f && __builtin_amdgcn_frexp_expf(af) < x - 21);
  };
  int xrun = -100;  // X of this wave's staged dims
  auto store_v = [&](int buf) __attribute__((always_inline)) {
    if constexpr (Q8) {
      // (what lies where no key is held may be another sequence's)
      const float fv = (dead >> lane) & 1 ? 0.0f : half_bits_to_float(vfr);
      const bool out = track(fv, xrun);
      if (lane == 0) vexp[wave] = xrun;
      if (out) left_out = 1;
      const _Float16 f = (_Float16)(out ? 0.0f : ldexpf(fv, 8 - xrun));
      const fh2 f2 = {f, f};
#pragma unroll
      for (int j = 0; j < PER; j++) {
        fh8 hi[2], lo[2];
#pragma unroll
        for (int w = 0; w < 4; w++) {
          fh2 a[2];
          int8_halves(vr[j][w], a[0], a[1]);
#pragma unroll
          for (int e = 0; e < 2; e++) {
            const fh2 p = a[e] * f2;
            const fh2 l = __builtin_elementwise_fma(a[e], f2, -p);  // the exact rest
            const int at = 4 * (w & 1) + 2 * e;
            hi[w >> 1][at] = p[0];
            hi[w >> 1][at + 1] = p[1];
            lo[w >> 1][at] = l[0];
            lo[w >> 1][at + 1] = l[1];
          }
        }
        const int pc = wave * (D / 32) + 2 * j;
#pragma unroll
        for (int e = 0; e < 2; e++) {
          const int at = lane * D + 8 * ((pc + e) ^ val_swz<D>(lane));
          *(fh8*)(vs[0] + at) = hi[e];
          *(fh8*)(vs[VH - 1] + at) = lo[e];
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < PER; j++) {
        const int i = tid + 256 * j, row = i / PIECES, pc = i % PIECES;
        *(fu4*)(vs[buf] + row * D + 8 * (pc ^ val_swz<D>(row))) = vr[j];
      }
    }
  };

  // the first slice on its way behind the queries, ahead of their conversion
  load(kc, s0, kr, kfr);
  load(vc, s0, vr, vfr);
  __builtin_amdgcn_sched_barrier(0);

  // The query, scaled by the power of two that brings its largest value to
  // [2^14, 2^15) and split into three halves; scores are taken against |scale|
  // log2(e), which takes the power back, the query carrying scale's sign.
  float c2 = fabsf(scale) * kLog2e;
  fh8 qf[3][D / 16];
  {
    float mx = 0.0f;
#pragma unroll
    for (int st = 0; st < D / 16; st++)
#pragma unroll
      for (int u = 0; u < 8; u++) mx = fmaxf(mx, fabsf(qraw[st][u >> 2][u & 3]));
    mx = other_max(mx);
    const int e = mx > 0.0f ? max(__builtin_amdgcn_frexp_expf(mx) - 15, -126) : 0;
    c2 = ldexpf(c2, e);
    const float sc = ldexpf(scale < 0.0f ? -1.0f : 1.0f, -e);
#pragma unroll
    for (int st = 0; st < D / 16; st++) {
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const float f = sc * qraw[st][u >> 2][u & 3];
        const _Float16 h1 = (_Float16)f;
        const float r1 = f - (float)h1;  // exact
        const _Float16 h2 = (_Float16)r1;
        qf[0][st][u] = h1;
        qf[1][st][u] = h2;
        qf[2][st][u] = (_Float16)(r1 - (float)h2);
      }
    }
  }

  ff16 o[NT];
#pragma unroll
  for (int dt = 0; dt < NT; dt++) o[dt] = ff16{};
  int xo[NT];  // q8_0: the X that o[dt] is held at
#pragma unroll
  for (int dt = 0; dt < NT; dt++) xo[dt] = -100;
  float mc = -1e30f, l = 0.0f;  // running maximum (of the scores, before c2) and this half wave's sum

  // Lane addresses in bytes.  A piece's slot is an exclusive or, and a row
  // starts at a multiple of the piece bits, so piece 2 st + h of this lane's
  // key (n of a tile) is at kat ^ (32 st), and the transposed read of dims
  // 32 dt + 16 b + 4 (i16 % 4) at rows 4 h + i16 / 4 (+ 8 v) of a 16-key step
  // at vat[v] ^ (64 dt).
  const int i16 = lane & 15, b16 = (lane >> 4) & 1;
  const uint32_t kat0 = 2 * n * D + 16 * (h ^ key_swz<D>(n));
  uint32_t vat0[2];
#pragma unroll
  for (int v = 0; v < 2; v++) {
    const int row = 4 * h + (i16 >> 2) + 8 * v;
    vat0[v] = 2 * row * D + 16 * ((2 * b16 + ((i16 & 3) >> 1)) ^ val_swz<D>(row)) + 8 * (i16 & 1);
  }
  typedef __attribute__((address_space(3))) const char* lds_ptr;
  const lds_ptr ks0 = (lds_ptr)&ks[0][0], vs0 = (lds_ptr)&vs[0][0];
  auto vfrag = [&](const uint32_t (&vat)[2], int dt, uint32_t at) __attribute__((always_inline)) {
    fs8 a;
#pragma unroll
    for (int v = 0; v < 2; v++) {
      const fs4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) fs4*)(vs0 + ((vat[v] ^ (64 * dt)) + at)));
#pragma unroll
      for (int e = 0; e < 4; e++) a[4 * v + e] = x[e];
    }
    return __builtin_bit_cast(fh8, a);
  };

  // 32 keys of slice sl: their scores, the running maximum and sum, the
  // weights' halves, and the weighted values
  auto tile = [&](int kt, int sl, int buf) __attribute__((always_inline)) {
    const int base = sl * kSlice + 32 * kt;
    // (opaque, so that the pieces' addresses are formed here and not kept in
    // registers across the loop, of which there are none to spare)
    uint32_t kat = kat0 + 2 * (buf * kSlice + 32 * kt) * D, vat[2] = {vat0[0], vat0[1]};
    asm volatile("" : "+v"(kat), "+v"(vat[0]), "+v"(vat[1]));
    typedef __attribute__((address_space(3))) const fh8* lds_h8;
    ff16 s = {};
    if constexpr (Q8) {
#pragma unroll
      for (int bl = 0; bl < NT; bl++) {
        ff16 c = {};
#pragma unroll
        for (int st = 2 * bl; st < 2 * bl + 2; st++) {
          const fh8 a = *(lds_h8)(ks0 + (kat ^ (32 * st)));
#pragma unroll
          for (int k = 0; k < 3; k++) c = mfma32(a, qf[k][st], c);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j4 = 0; j4 < 4; j4++) {
          const ff4 f = *(const ff4*)&kf[buf][bl][32 * kt + 8 * j4 + 4 * h];
#pragma unroll
          for (int e = 0; e < 4; e++) s[4 * j4 + e] = fmaf(f[e], c[4 * j4 + e], s[4 * j4 + e]);
        }
      }
    } else {
#pragma unroll
      for (int st = 0; st < D / 16; st++) {
        const fh8 a = *(lds_h8)(ks0 + (kat ^ (32 * st)));
#pragma unroll
        for (int k = 0; k < 3; k++) s = mfma32(a, qf[k][st], s);
        if (st & 1) __builtin_amdgcn_sched_barrier(0);
      }
    }
    // lanes past their token's end, or on a cell that is not held, take no part
    const bool full = !PAGED && base + 32 <= wave_min;
    const int rel = cnt - base - 4 * h;
    uint32_t held = 0xffffffffu;
    if constexpr (PAGED) held = (uint32_t)__ballot(kv_index[min(base + n, count - 1)] >= 0) >> (4 * h);
    auto live = [&](int j) __attribute__((always_inline)) {
      const int at = 8 * (j >> 2) + (j & 3);
      return at < rel && (!PAGED || ((held >> at) & 1));
    };
    if (!full) {
#pragma unroll
      for (int j = 0; j < 16; j++) s[j] = live(j) ? s[j] : -INFINITY;
    }
    float m = s[0];
#pragma unroll
    for (int j = 1; j < 16; j++) m = fmaxf(m, s[j]);
    m = other_max(m);
    const float mn = fmaxf(mc, m);
    if (__any(mn != mc)) {
      const float a = __builtin_amdgcn_exp2f((mc - mn) * c2);
      l *= a;
#pragma unroll
      for (int dt = 0; dt < NT; dt++) o[dt] *= a;
      mc = mn;
    }
    fh8 ph[2], pl[2];
#pragma unroll
    for (int j = 0; j < 16; j++) {
      // (the difference first: at scores of 1e9 c2 mc is rounded by up to 64,
      // and a weight taken against it overflows a half)
      float p = __builtin_amdgcn_exp2f((s[j] - mc) * c2);
      if (!full) p = live(j) ? p : 0.0f;
      l += p;
      const _Float16 hi = (_Float16)fmaf(p, kLift, 0.0f);  // (one instruction)
      ph[j >> 3][j & 7] = hi;
      pl[j >> 3][j & 7] = (_Float16)fmaf(p, kLift, -(float)hi);
    }
    if constexpr (Q8) {
#pragma unroll
      for (int dt = 0; dt < NT; dt++) {
        const int x = __builtin_amdgcn_readfirstlane(vexp[dt * 32 / (D / 4)]);
        if (x != xo[dt]) {
          o[dt] *= ldexpf(1.0f, xo[dt] - x);
          xo[dt] = x;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int dt = 0; dt < NT; dt++) {
        const fh8 a = vfrag(vat, dt, 2 * ((Q8 ? 0 : buf * kSlice) + 32 * kt + 16 * u) * D);
        o[dt] = mfma32(a, ph[u], o[dt]);
        o[dt] = mfma32(a, pl[u], o[dt]);
        if constexpr (Q8) o[dt] = mfma32(vfrag(vat, dt, 2 * (kSlice + 32 * kt + 16 * u) * D), ph[u], o[dt]);
        if (dt & 1) __builtin_amdgcn_sched_barrier(0);
      }
  };

  store_k(0);
  store_v(0);
  __syncthreads();
  for (int sl = s0; sl < s1; sl++) {
    const int buf = (sl - s0) & 1, base = sl * kSlice;
    const bool more = sl + 1 < s1;          // uniform
    const bool mine = base < wave_max;      // this wave has tokens that reach the slice
    if (more) load(kc, sl + 1, kr, kfr);
    // the slice's weights, 32 keys at a time (both tiles' scores at once are 32
    // more registers than a wave has)
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      if (mine && base + 32 * kt < wave_max) tile(kt, sl, buf);
      if (kt == 0 && more) {
        store_k(1 - buf);
        int next = sl + 1;
        asm volatile("" : "+s"(next));  // (the keys' row offsets are not kept for it)
        load(vc, next, vr, vfr);
      }
    }
    if (Q8) __syncthreads();  // the one value buffer has been read
    if (more) store_v(1 - buf);
    __syncthreads();
  }

  // q8_0: the keys that were left out (the same ones: X runs as it did), added
  // in float32 to the rows that they are live for.  Their weights are in l.
  if constexpr (Q8) {
    if (__builtin_expect(left_out, 0)) {
      // (from the thread's index again, and the queries' power of two out of c2:
      // kept through the loop they cost it six registers, which it spilled)
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));
      const int lane = tid & 63, h = lane >> 5, r = 32 * (tid >> 6) + (lane & 31);
      const int t = t0 + r / group, head = kvh * group + r % group, cnt = t < tokens ? pos[t] + 1 : 0;
      const int e = __builtin_amdgcn_frexp_expf(c2) - __builtin_amdgcn_frexp_expf(fabsf(scale) * kLog2e);
      const float sc = ldexpf(scale < 0.0f ? -1.0f : 1.0f, -e);
      const float* qr = q + (int64_t)min(t, tokens - 1) * q_stride + (int64_t)head * D + 8 * h;
#pragma unroll
      for (int dt = 0; dt < NT; dt++) {
        int x = -100;
        for (int sl = s0; sl < s1; sl++) {
          const int cell = cell_of(sl, lane);
          float f = __half2float(vc[row_of(cell) + (kvw >> 1) + ((kvh * D) >> 5) + dt]);
          if (sl * kSlice + lane >= count || cell < 0) f = 0.0f;
          for (uint64_t outs = __ballot(track(f, x)); outs; outs &= outs - 1) {
            const int k = __builtin_ctzll(outs);
            const int64_t row = row_of(__shfl(cell, k));
            const int8_t* kb = (const int8_t*)(kc + row) + kvh * D + 8 * h;
            const __half* kfac = kc + row + (kvw >> 1) + ((kvh * D) >> 5);
            float s = 0.0f;
#pragma nounroll
            for (int st = 0; st < D / 16; st++) {
              float b = 0.0f;
              for (int u = 0; u < 8; u++) b = fmaf((float)kb[16 * st + u], sc * qr[16 * st + u], b);
              s = fmaf(__half2float(kfac[st >> 1]), b, s);
            }
            s = other_sum(s);
            const float p = __builtin_amdgcn_exp2f((s - mc) * c2) * kLift;
            const float fk = __shfl(f, k) * ldexpf(1.0f, 8 - xo[dt]);
            const int8_t* vb = (const int8_t*)(vc + row) + kvh * D + 32 * dt + 4 * h;
            if (sl * kSlice + k < cnt) {
#pragma unroll
              for (int j = 0; j < 16; j++)
                o[dt][j] = fmaf(p, (float)vb[8 * (j >> 2) + (j & 3)] * fk, o[dt][j]);
            }
          }
        }
      }
    }
  }

  l = other_sum(l);
  if (!live_row) return;
  const int64_t rowi = (int64_t)t * heads + head;
  float* dst = splits == 1 ? out + rowi * D : part_acc + (rowi * splits + split) * D;
  const float w = (splits == 1 ? 1.0f / l : 1.0f) * (1.0f / kLift);
#pragma unroll
  for (int dt = 0; dt < NT; dt++) {
    const float f = Q8 ? w * ldexpf(1.0f, xo[dt] - 8) : w;
#pragma unroll
    for (int j4 = 0; j4 < 4; j4++) {
      ff4 v;
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = o[dt][4 * j4 + e] * f;
      *(ff4*)(dst + 32 * dt + 8 * j4 + 4 * h) = v;
    }
  }
  if (splits > 1 && h == 0) *(float2*)(part_ml + (rowi * splits + split) * 2) = make_float2(mc * c2, l);
}

// Folds the splits of each (token, head) row: thread = 4 dims.  A split that
// no key of the row falls in has sum 0 and is left out.
template <int D>
__global__ __launch_bounds__(256) void attend_combine_kernel(const float* __restrict__ part_acc,
                                                             const float* __restrict__ part_ml, int rows, int splits,
                                                             float* __restrict__ out) {
  constexpr int TPR = D / 4;
  const int row = blockIdx.x * (256 / TPR) + threadIdx.x / TPR, d4 = threadIdx.x % TPR;
  if (row >= rows) return;
  const float2* ml = (const float2*)part_ml + (int64_t)row * splits;
  const ff4* acc = (const ff4*)(part_acc + (int64_t)row * splits * D) + d4;
  float m = -INFINITY;
  for (int s = 0; s < splits; s++) {
    const float2 v = ml[s];
    if (v.y != 0.0f) m = fmaxf(m, v.x);
  }
  ff4 o = {0.0f, 0.0f, 0.0f, 0.0f};
  float l = 0.0f;
#pragma unroll 4
  for (int s = 0; s < splits; s++) {
    const float2 v = ml[s];
    const ff4 a = acc[s * TPR];
    if (v.y != 0.0f) {
      const float w = __builtin_amdgcn_exp2f(v.x - m);
      l = fmaf(v.y, w, l);
#pragma unroll
      for (int e = 0; e < 4; e++) o[e] = fmaf(a[e], w, o[e]);
    }
  }
  const float w = 1.0f / l;
  ((ff4*)out)[(int64_t)row * TPR + d4] = o * w;
}

// Shares of the keys: enough that the blocks fill two a compute unit, at
// most one for each slice of the context, and at most 16 (each is another
// partial result of every row to write and fold).
int flash_splits(int kv_heads, int tiles, int max_count) {
  const int slices = (max_count + kSlice - 1) / kSlice;
  const int want = 2 * cu_count() / std::max(1, kv_heads * tiles);
  return std::max(1, std::min({want, slices, 16}));
}

}  // namespace

bool flash_fits(int32_t heads, int32_t kv_heads, int32_t head_dim, int32_t tokens) {
  const int group = heads / kv_heads;
  return tokens > kMaxTokens && (head_dim == 64 || head_dim == 128) &&
         (group == 1 || group == 2 || group == 4 || group == 8);
}

int launch_attend_flash(hipStream_t s, const float* q, int64_t q_stride, const uint16_t* k_cache,
                        const uint16_t* v_cache, int32_t heads, int32_t kv_heads, int32_t head_dim, float scale,
                        const int32_t* pos, int32_t max_count, int32_t tokens, float* out, float* part_acc,
                        float* part_ml, int32_t form, const int32_t* kv_index) {
  const int group = heads / kv_heads, tq = kRows / group, tiles = (tokens + tq - 1) / tq;
  const int splits = flash_splits(kv_heads, tiles, max_count);
  const int row = cache_row(form, kv_heads * head_dim);
  const dim3 grid(splits, kv_heads, tiles);
#define MI_FLASH(DD, Q, P)                                                                                       \
  hipLaunchKernelGGL((attend_flash_kernel<DD, Q, P>), grid, dim3(256), 0, s, q, q_stride, (const __half*)k_cache, \
                     (const __half*)v_cache, row, heads, kv_heads, group, scale, pos, tokens, kv_index, part_acc, \
                     part_ml, out)
#define MI_FLASH_F(DD)                         \
  if (form == MI_CACHE_Q8) {                   \
    if (kv_index) MI_FLASH(DD, true, true);    \
    else MI_FLASH(DD, true, false);            \
  } else {                                     \
    if (kv_index) MI_FLASH(DD, false, true);   \
    else MI_FLASH(DD, false, false);           \
  }
  if (head_dim == 64) {
    MI_FLASH_F(64)
  } else {
    MI_FLASH_F(128)
  }
#undef MI_FLASH_F
#undef MI_FLASH
  int rc = hip_check(hipGetLastError(), "attend_flash launch");
  if (rc || splits == 1) return rc;
  const int rows = tokens * heads, rpb = 256 / (head_dim / 4);
  if (head_dim == 64)
    hipLaunchKernelGGL(attend_combine_kernel<64>, dim3((rows + rpb - 1) / rpb), dim3(256), 0, s, part_acc, part_ml, rows,
                       splits, out);
  else
    hipLaunchKernelGGL(attend_combine_kernel<128>, dim3((rows + rpb - 1) / rpb), dim3(256), 0, s, part_acc, part_ml, rows,
                       splits, out);
  return hip_check(hipGetLastError(), "attend_combine launch");
}

}  // namespace mi
