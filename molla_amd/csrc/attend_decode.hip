// attend_decode.hip -- decode attention on the matrix cores
// (v_mfma_f32_16x16x32_f16), gfx950: attention.mojo:144 attend for one query
// token per sequence, over an f16 or a q8_0 cache (gpu_ops.mojo:678
// attend_kernel's `form`), GQA with up to 8 query heads a key head, head_dim
// 64 or 128; the split and the fold of gpu_ops.mojo:929 / 1104.
//
// A block takes a share of one (key head, token)'s keys: every shares-th step of
// 32 keys a wave.  Each of its two or four waves walks its 32-key runs by itself,
// with a running maximum and sum in registers and its own LDS rows for the values
// (no block barrier until the waves' results are folded at the end), and sends for
// the next run's keys and values as soon as it has used this one's.  The number of
// shares (decode_attend_plan) is the one with the fewest runs in line on a compute
// unit, at most 64, so a long context costs a few partial results a head and
// not one a 64-key slice.
//
// What bounds it: to about 1000 keys a chain of latencies (cycles of a block with
// one run a wave: the position ~1000, the keys ~2500, the softmax ~800, the values
// to LDS ~400, the weighted values ~700, then the fold); beyond, the loads.  us of
// a layer of width 256 with 32 heads of 128 over 8 key heads, caches cold (a 64-key
// slice a block and a merge of the slices -> now): one sequence of 300 keys 26.2 ->
// 26.4, of 2304 28.6 -> 28.3, of 32768 71.2 -> 51.1; eight of 300 50.9 -> 50.5, of
// 2304 64.7 -> 64.6, of 8000 102.7 -> 96.4; eight of 6000 and less, paged q8_0, 101.5
// -> 79.5.
//
//   S^T = K Q^T, keys as rows (read straight from the cache) and queries as
//   columns: a lane's 8 scores belong to its own query, the softmax takes two
//   exchanges between lanes, and the weights are in place as the B operand of
//   O^T = V^T P^T.  Queries enter as three halves, scaled to their largest value
//   (as in attend_flash.hip), P as two after a lift by 2^14; values lie by rows
//   in LDS and are read transposed (ds_read_b64_tr_b16).  Slot i of lane group
//   g takes key 4 g + i % 4 + 16 (i / 4), the order in which S^T leaves them.
//
// q8_0: quants enter as exact halves; a key block's factor multiplies its part
// of the score, a value block's the weights.  The products enter as two halves,
// scaled by 2^(15 - X) with X the exponent of the column's largest one since its
// maximum last rose: to 2^-39 of that, whatever the factors' range.  A key that
// is not there has a factor of 0.
//
// MFMA fragments (16x16x32): lane l holds row / column l % 16 and values
// 8 (l / 16) .. +8 of the 32; result element i of lane l is row 4 (l / 16) +
// i, column l % 16.
#include <math.h>

#include <algorithm>

#include "mi_internal.h"

namespace mi {
namespace {

typedef _Float16 dh2 __attribute__((ext_vector_type(2)));
typedef _Float16 dh8 __attribute__((ext_vector_type(8)));
typedef short ds4 __attribute__((ext_vector_type(4)));
typedef short ds8 __attribute__((ext_vector_type(8)));
typedef float df4 __attribute__((ext_vector_type(4)));
typedef uint32_t du4 __attribute__((ext_vector_type(4)));
typedef uint32_t du2 __attribute__((ext_vector_type(2)));

constexpr int kRun = 32;            // keys a wave takes at a time
constexpr int kMaxShares = 64;      // of a (key head, token)'s keys
constexpr float kLift = 16384.0f;   // of P when it is split: see attend_flash.hip
constexpr float kLog2e = 1.44269504088896340736f;

__device__ __forceinline__ df4 mfma16(dh8 a, dh8 b, df4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// 16-byte piece pc of LDS row r lies at slot pc ^ swz(r): a transposed read
// takes 4 rows x 32 bytes per 16 lanes, on distinct banks.
template <int D>
__device__ __forceinline__ int swz(int r) {
  return (D == 128 ? 4 * (r & 3) : 4 * ((r >> 1) & 1)) | ((r >> 2) & 3);
}

// over the four lanes that share a column
template <class Op>
__device__ __forceinline__ float across(float v, Op op) {
  auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = op(__uint_as_float(p[0]), __uint_as_float(p[1]));
  p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return op(__uint_as_float(p[0]), __uint_as_float(p[1]));
}

__device__ __forceinline__ dh2 as_dh2(uint32_t u) { return __builtin_bit_cast(dh2, u); }

// eight signed bytes as halves: 0x64 above byte + 128 is 1152 + byte
__device__ __forceinline__ dh8 int8_halves(uint32_t x, uint32_t y) {
  const dh2 off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
  x ^= 0x80808080u;
  y ^= 0x80808080u;
  const du4 m = {__builtin_amdgcn_perm(0x64646464u, x, 0x04010400u), __builtin_amdgcn_perm(0x64646464u, x, 0x04030402u),
                 __builtin_amdgcn_perm(0x64646464u, y, 0x04010400u), __builtin_amdgcn_perm(0x64646464u, y, 0x04030402u)};
  du4 r;
#pragma unroll
  for (int i = 0; i < 4; i++) r[i] = __builtin_bit_cast(uint32_t, as_dh2(m[i]) + off);
  return __builtin_bit_cast(dh8, r);
}

// The grid is (shares, kv_heads, tokens); share s takes every shares-th step of
// 32 keys a wave of the token's own count (a device value: the host knows only
// the context), starting at the s-th, and writes each head's unnormalised sum
// with (maximum, sum) in base 2 to slot (token, head, share); (0, 0) for no
// keys.
template <int D, bool Q8, bool PAGED, int W>
__global__ __launch_bounds__(64 * W, 2) void attend_decode_kernel(
    const float* __restrict__ q, int64_t q_stride, const __half* __restrict__ kc, const __half* __restrict__ vc,
    int64_t cache_stride, int row_halves, int heads, int kv_heads, int group, float scale,
    const int32_t* __restrict__ pos, int count_host, const int32_t* __restrict__ kv_index, int64_t index_stride,
    float* __restrict__ part_acc, float* __restrict__ part_ml) {
  constexpr int kStep = kRun * W;  // keys a block takes at a time
  constexpr int KS = D / 32, NT = D / 16, PIECES = D / 8;
  constexpr int kFac = Q8 ? 2 * KS * kRun : 1;             // floats: factors of a run's keys and values
  constexpr int kWaveBytes = kRun * D * 2;                 // a run's values as halves
  __shared__ __align__(16) uint8_t vs[W][kWaveBytes];      // afterwards the waves' sums
  __shared__ __align__(16) float fac[W][kFac];
  __shared__ __align__(16) float wml[2][8][W];  // (maximum, sum) of a head, the waves side by side
  static_assert(8 * D * 4 <= kWaveBytes, "a wave's sums of 8 heads in place of its values");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lm = lane & 15, lk = lane >> 4;
  const int share = blockIdx.x, shares = gridDim.x, kvh = blockIdx.y, t = blockIdx.z;
  const int64_t slot0 = ((int64_t)t * heads + (int64_t)kvh * group) * shares + share;
  const int count = pos ? pos[t] + 1 : count_host;
  // the queries, first in line, also ahead of the position: column lm (past the
  // group, the last one)
  const float* qr = q + (int64_t)t * q_stride + ((int64_t)kvh * group + min(lm, group - 1)) * D + 8 * lk;
  df4 qraw[KS][2];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    qraw[ks][0] = *(const df4*)(qr + 32 * ks);
    qraw[ks][1] = *(const df4*)(qr + 32 * ks + 4);
  }
  __builtin_amdgcn_sched_barrier(0);
  if (share * kStep >= count) {
    if (tid < group) *(float2*)(part_ml + (slot0 + (int64_t)tid * shares) * 2) = make_float2(0.0f, 0.0f);
    return;
  }
  if (PAGED) kv_index += t * index_stride;
  const int64_t seq = PAGED ? 0 : (int64_t)t * cache_stride;
  const int kvw = kv_heads * D;
  // The cells of a run's keys, key lane % 32 a lane (keys past the end repeat
  // the last one, masked below): read a run ahead of its keys and values, which
  // take theirs from the lane that has it
  auto cells_of = [&](int key) __attribute__((always_inline)) {
    const int j = min(key + (lane & 31), count - 1);
    return PAGED ? kv_index[j] : j;
  };
  auto row_of = [&](int key, int cells, int r) __attribute__((always_inline)) {
    const int cell = PAGED ? max(__shfl(cells, r), 0) : min(key + r, count - 1);
    return seq + (int64_t)cell * row_halves;
  };

  // a run's keys (lane: key lm of each 16-key tile, its values 32 ks + 8 lk ..
  // +8), values (16-byte pieces of its rows) and q8_0 factors (lane: key
  // lane % 32, keys' below lane 32 and values' above)
  typedef typename std::conditional<Q8, du2, du4>::type KWord;
  constexpr int VW = Q8 ? kRun * D / 16 / 64 : kRun * PIECES / 64;
  KWord kw[2][KS];
  du4 vw[VW];
  du2 fw = {0, 0};
  auto load_k = [&](int key0, int cells) __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < 2; a++) {
      const __half* r = kc + row_of(key0, cells, 16 * a + lm);
#pragma unroll
      for (int ks = 0; ks < KS; ks++)
        kw[a][ks] = Q8 ? *(const KWord*)((const int8_t*)r + kvh * D + 32 * ks + 8 * lk)
                       : *(const KWord*)(r + kvh * D + 32 * ks + 8 * lk);
    }
  };
  auto load_v = [&](int key0, int cells) __attribute__((always_inline)) {
    if constexpr (Q8) {
      const __half* c = (lane < 32 ? kc : vc) + row_of(key0, cells, lane & 31) + (kvw >> 1) + ((kvh * D) >> 5);
      if constexpr (KS == 4) fw = *(const du2*)c;
      else fw.x = *(const uint32_t*)c;
    }
#pragma unroll
    for (int j = 0; j < VW; j++) {
      const int i = lane + 64 * j;
      if constexpr (Q8) vw[j] = *(const du4*)((const int8_t*)(vc + row_of(key0, cells, i / (D / 16))) + kvh * D + 16 * (i % (D / 16)));
      else vw[j] = *(const du4*)(vc + row_of(key0, cells, i / PIECES) + kvh * D + 8 * (i % PIECES));
    }
  };
  df4 o[NT];
#pragma unroll
  for (int dt = 0; dt < NT; dt++) o[dt] = df4{0.0f, 0.0f, 0.0f, 0.0f};
  int xo[Q8 ? KS : 1];  // q8_0: the X that this column's 32-dim blocks of o are held at
#pragma unroll
  for (int b = 0; b < (Q8 ? KS : 1); b++) xo[b] = -100;
  // this wave's maximum in base 2 and sum
  float m2 = -INFINITY, l = 0.0f;

  const int stride = shares * kStep;  // to this wave's next run
  int key0 = share * kStep + kRun * wave;
  if (key0 < count) {  // (uniform over the wave; else it has no keys)
    int cells = cells_of(key0);
    load_k(key0, cells);
    load_v(key0, cells);
    int cells_next = cells_of(key0 + stride);
    __builtin_amdgcn_sched_barrier(0);

    // the queries as B fragments: column lm (zero past the group), each scaled by
    // a power of two that c2 takes back (as in attend_flash.hip)
    float c2 = fabsf(scale) * kLog2e;
    dh8 qf[3][KS];
    {
      float mx = 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS; ks++)
#pragma unroll
        for (int u = 0; u < 8; u++) mx = fmaxf(mx, fabsf(qraw[ks][u >> 2][u & 3]));
      mx = across(mx, lanes::Max{});
      const int e = mx > 0.0f ? max(__builtin_amdgcn_frexp_expf(mx) - 15, -126) : 0;
      c2 = ldexpf(c2, e);
      const float sc = lm < group ? ldexpf(scale < 0.0f ? -1.0f : 1.0f, -e) : 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
#pragma unroll
        for (int u = 0; u < 8; u++) {
          const float f = qraw[ks][u >> 2][u & 3] * sc;
          const _Float16 h1 = (_Float16)f;
          const float r1 = fmaf((float)h1, -1.0f, f);  // exact (as an fma it takes the half as it is)
          const _Float16 h2 = (_Float16)r1;
          qf[0][ks][u] = h1;
          qf[1][ks][u] = h2;
          qf[2][ks][u] = (_Float16)fmaf((float)h2, -1.0f, r1);
        }
      }
    }

    typedef __attribute__((address_space(3))) char* lds_ptr;
    const lds_ptr vl = (lds_ptr)&vs[wave][0];
    float* fl = fac[wave];
    // transposed reads: rows 4 lk + i16 / 4 (+ 16), dims 16 dt + 4 (i16 % 4): the
    // slot is an exclusive or with bits a row's start leaves free
    uint32_t vat[2];
#pragma unroll
    for (int v = 0; v < 2; v++) {
      const int row = 4 * lk + (lm >> 2) + 16 * v;
      vat[v] = 2 * row * D + 16 * (((lm & 3) >> 1) ^ swz<D>(row)) + 8 * (lm & 1);
    }
    float mc = -1e30f;  // the running maximum, of the scores before c2

    for (; key0 < count; key0 += stride) {  // (uniform over the wave)
      uint32_t held = 0xffffffffu;
      if constexpr (PAGED) held = (uint32_t)__ballot(cells >= 0);
      const int nk = min(kRun, count - key0);
      if (nk < kRun) held &= (1u << nk) - 1u;
      df4 s[2];
      if constexpr (Q8) {
        // factors to LDS by (key | value, block, key), read back four keys a
        // lane; zero for a key past the end or not held, whose row is another's
        if (!((held >> (lane & 31)) & 1)) fw = du2{0, 0};
#pragma unroll
        for (int b = 0; b < KS; b++)
          fl[(lane >> 5) * KS * kRun + b * kRun + (lane & 31)] = half_bits_to_float(b < 2 ? fw.x >> (16 * b) : fw.y >> (16 * (b - 2)));
        asm volatile("" ::: "memory");
#pragma unroll
        for (int a = 0; a < 2; a++) {
          s[a] = df4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int ks = 0; ks < KS; ks++) {
            const dh8 k8 = int8_halves(kw[a][ks].x, kw[a][ks].y);
            df4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int h = 0; h < 3; h++) c = mfma16(k8, qf[h][ks], c);
            const df4 f = *(const df4*)(fl + ks * kRun + 16 * a + 4 * lk);
#pragma unroll
            for (int i = 0; i < 4; i++) s[a][i] = fmaf(f[i], c[i], s[a][i]);
          }
        }
      } else {
#pragma unroll
        for (int a = 0; a < 2; a++) {
          s[a] = df4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int h = 0; h < 3; h++) s[a] = mfma16(__builtin_bit_cast(dh8, kw[a][ks]), qf[h][ks], s[a]);
        }
      }
      const bool more = key0 + stride < count;  // uniform
      if (more) load_k(key0 + stride, cells_next);

      // running maximum and weights of this lane's keys 16 a + 4 lk + i
      const uint32_t mine = held >> (4 * lk);
      float m = -INFINITY;
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          s[a][i] = (mine >> (16 * a + i)) & 1 ? s[a][i] : -INFINITY;
          m = fmaxf(m, s[a][i]);
        }
      m = across(m, lanes::Max{});
      const float mn = fmaxf(mc, m);
      const bool rose = mn != mc;
      if (__any(rose && l != 0.0f)) {  // (else there is nothing yet)
        const float f = __builtin_amdgcn_exp2f((mc - mn) * c2);
        l *= f;
#pragma unroll
        for (int dt = 0; dt < NT; dt++) o[dt] *= f;
      }
      mc = mn;
      float p[8];
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float e = __builtin_amdgcn_exp2f((s[a][i] - mc) * c2);  // (as in attend_flash.hip)
          p[4 * a + i] = (mine >> (16 * a + i)) & 1 ? e : 0.0f;
          l += p[4 * a + i];
        }

      // the values to this wave's LDS rows
#pragma unroll
      for (int j = 0; j < VW; j++) {
        const int i = lane + 64 * j;
        if constexpr (Q8) {
          const int row = i / (D / 16), pc = 2 * (i % (D / 16));
          *(__attribute__((address_space(3))) dh8*)(vl + 2 * row * D + 16 * (pc ^ swz<D>(row))) = int8_halves(vw[j].x, vw[j].y);
          *(__attribute__((address_space(3))) dh8*)(vl + 2 * row * D + 16 * ((pc + 1) ^ swz<D>(row))) = int8_halves(vw[j].z, vw[j].w);
        } else {
          const int row = i / PIECES, pc = i % PIECES;
          *(__attribute__((address_space(3))) du4*)(vl + 2 * row * D + 16 * (pc ^ swz<D>(row))) = vw[j];
        }
      }
      df4 fv[Q8 ? KS : 1][2];
      if constexpr (Q8) {
#pragma unroll
        for (int b = 0; b < KS; b++)
#pragma unroll
          for (int a = 0; a < 2; a++) fv[b][a] = *(const df4*)(fl + KS * kRun + b * kRun + 16 * a + 4 * lk);
      }
      asm volatile("" ::: "memory");  // (a wave's LDS operations complete in order)
      if (more) load_v(key0 + stride, cells_next);
      cells = cells_next;
      cells_next = cells_of(key0 + 2 * stride);

      dh8 ph, pl;
      if constexpr (!Q8) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
          ph[i] = (_Float16)fmaf(p[i], kLift, 0.0f);  // (one instruction)
          pl[i] = (_Float16)fmaf(p[i], kLift, -(float)ph[i]);
        }
      }
#pragma unroll
      for (int dt = 0; dt < NT; dt++) {
        if constexpr (Q8) {
          if (dt % 2 == 0) {
            const int b = dt / 2;
            float w[8], wm = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; i++) {
              w[i] = p[i] * fv[b][i >> 2][i & 3];
              wm = fmaxf(wm, fabsf(w[i]));
            }
            wm = across(wm, lanes::Max{});
            // (an infinite factor: the finite products are below 2^31)
            const int xw = wm < INFINITY ? __builtin_amdgcn_frexp_expf(wm) : 31;
            const int x = wm > 0.0f ? max(max(xw, rose ? xo[b] - 60 : xo[b]), -100) : xo[b];
            if (__any(x != xo[b])) {
              const float f = ldexpf(1.0f, xo[b] - x);
              o[dt] *= f;
              o[dt + 1] *= f;
              xo[b] = x;
            }
            const float unit = ldexpf(1.0f, 15 - x);
#pragma unroll
            for (int i = 0; i < 8; i++) {
              const float v = w[i] * unit;
              ph[i] = (_Float16)v;
              pl[i] = (_Float16)(v - (float)ph[i]);
            }
            if (__builtin_expect(__any(!(wm < INFINITY)), 0)) {
#pragma unroll
              for (int i = 0; i < 8; i++)
                if (!(fabsf(w[i]) < INFINITY)) pl[i] = 0;
            }
          }
        }
        ds8 a;
#pragma unroll
        for (int v = 0; v < 2; v++) {
          const ds4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) ds4*)(vl + (vat[v] ^ (32 * dt))));
#pragma unroll
          for (int e = 0; e < 4; e++) a[4 * v + e] = x[e];
        }
        o[dt] = mfma16(__builtin_bit_cast(dh8, a), ph, o[dt]);
        o[dt] = mfma16(__builtin_bit_cast(dh8, a), pl, o[dt]);
      }
      asm volatile("" ::: "memory");  // the reads above stay ahead of the next run's stores
    }
    l = across(l, lanes::Add{});
    if (l != 0.0f) m2 = mc * c2;  // (no key held: no part in the fold)
  }

  // fold the waves: their sums (in place of the values) and (maximum, sum), four
  // dims a thread and every read sent for at once (a dim at a time, with the
  // weights found again for each, this took 3700 of a short context's 10000
  // cycles)
  float* wo = (float*)&vs[0][0];  // [wave][group][D]
  __syncthreads();
  if (lm < group) {
#pragma unroll
    for (int dt = 0; dt < NT; dt++) {
      if constexpr (Q8) o[dt] *= ldexpf(1.0f, xo[dt / 2] - 15);
      *(df4*)(wo + (wave * group + lm) * D + 16 * dt + 4 * lk) = o[dt];
    }
    if (lk == 0) {
      wml[0][lm][wave] = m2;
      wml[1][lm][wave] = l;
    }
  }
  __syncthreads();
  for (int i = tid; i < group * (D / 4); i += 64 * W) {
    const int g = i / (D / 4), d = 4 * (i % (D / 4));
    df4 a[W];
    float mw[W], lw[W], m = -3e38f;
#pragma unroll
    for (int w = 0; w < W; w++) {
      a[w] = *(const df4*)(wo + (w * group + g) * D + d);
      mw[w] = wml[0][g][w];
      lw[w] = wml[1][g][w];
      m = fmaxf(m, mw[w]);
    }
    df4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < W; w++) {
      const float f = __builtin_amdgcn_exp2f(mw[w] - m);
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = fmaf(a[w][e], f, v[e]);
      sum = fmaf(lw[w], f, sum);
    }
    const int64_t slot = slot0 + (int64_t)g * shares;
    *(df4*)(part_acc + slot * D + d) = Q8 ? v : v * (1.0f / kLift);
    if (d == 0) *(float2*)(part_ml + slot * 2) = make_float2(m, sum);
  }
}

}  // namespace

bool decode_attend_fits(int32_t group, int32_t head_dim) {
  return (group == 1 || group == 2 || group == 4 || group == 8) && (head_dim == 64 || head_dim == 128);
}

// Two-wave blocks while every 64 keys of the context can have a compute unit of
// their own: one unit takes in about 64 bytes a cycle, so that a short context is
// better spread (us of a layer of width 256, two / four waves: 300 keys 26.3 / 27.4,
// 700 in a context of 1024 26.9 / 27.7, 1100 in 2048 27.6 / 28.0, four sequences of
// 300 in 512 38.3 / 39.6, two of 600 in 1024, q8_0, 40.3 / 39.8; past the line eight
// of 300 in 512 51.4 / 50.5, one of 2304 28.7 / 28.2).
//
// Shares: a compute unit with n blocks of r runs a wave takes n r runs' time, whether
// the blocks run side by side or in turn, and about a quarter of a run's for each
// block (us as above; 2304 keys, 18 steps, 32 pairs of a token and a key head: 6
// shares of 3 are 192 blocks and 46.1, 9 of 2 are 288 and 49.3, 18 of 1 are 576 and
// 46.9; 64 pairs: 4 shares 64.6, 6 64.8, 8 66.3, 16 69.9).  The fold takes another
// 1/128 of a run's for each share (one q8_0 sequence of 9000 in a context of 16384:
// 32 shares 35.2, 64 38.0).  q8_0's loads wait on more arithmetic, so that one block
// a unit is a little slower than that (eight paged sequences of 6000: 4 shares 86.3,
// 8 78.7, 16 83.0; two of 9000: 16 shares 52.8, 32 54.2).  At most 64 shares, which
// the fold takes in one round.
DecodePlan decode_attend_plan(int32_t kv_heads, int32_t tokens, int32_t max_count, bool q8) {
  const int64_t pairs = (int64_t)kv_heads * tokens, cus = cu_count();
  const int waves = pairs * ((max_count - 1) / (2 * kRun) + 1) <= cus ? 2 : 4;
  const int64_t steps = (max_count - 1) / (kRun * waves) + 1;
  DecodePlan best{waves, 1};
  int64_t least = INT64_MAX;
  for (int n = 1; n <= std::min<int64_t>(steps, kMaxShares); n++) {
    const int64_t deep = (n * pairs + cus - 1) / cus;
    int64_t cost = 16 * deep * (4 * ((steps + n - 1) / n) + 1) + n / 2;
    if (q8 && deep == 1) cost += cost / 32;
    if (cost < least) best.shares = n, least = cost;
  }
  return best;
}

int launch_attend_decode(hipStream_t s, const float* q, int64_t q_stride, const uint16_t* k_cache,
                         const uint16_t* v_cache, int64_t cache_stride, int32_t heads, int32_t kv_heads,
                         int32_t head_dim, float scale, const int32_t* pos, int32_t count_host, DecodePlan plan,
                         int32_t tokens, float* part_acc, float* part_ml, int32_t form, const int32_t* kv_index,
                         int64_t index_stride) {
  const int row = cache_row(form, kv_heads * head_dim);
  const dim3 grid(plan.shares, kv_heads, tokens);
#define MI_DEC_W(DD, Q, P, W)                                                                                      \
  hipLaunchKernelGGL((attend_decode_kernel<DD, Q, P, W>), grid, dim3(64 * W), 0, s, q, q_stride,                   \
                     (const __half*)k_cache, (const __half*)v_cache, cache_stride, row, heads, kv_heads,           \
                     heads / kv_heads, scale, pos, count_host, kv_index, index_stride, part_acc, part_ml)
#define MI_DEC(DD, Q, P)                              \
  if (plan.waves == 4) MI_DEC_W(DD, Q, P, 4);         \
  else MI_DEC_W(DD, Q, P, 2);
#define MI_DEC_F(DD)                         \
  if (form == MI_CACHE_Q8) {                 \
    if (kv_index) { MI_DEC(DD, true, true) }    \
    else { MI_DEC(DD, true, false) }            \
  } else {                                   \
    if (kv_index) { MI_DEC(DD, false, true) }   \
    else { MI_DEC(DD, false, false) }           \
  }
  if (head_dim == 64) {
    MI_DEC_F(64)
  } else {
    MI_DEC_F(128)
  }
#undef MI_DEC_F
#undef MI_DEC
#undef MI_DEC_W
  return hip_check(hipGetLastError(), "attend_decode launch");
}

}  // namespace mi
