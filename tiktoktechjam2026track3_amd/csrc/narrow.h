// Device pieces of the narrow-model kernels (d_model and ffn_dim of 32, 64 or
// 128): a wavefront owns 16 tokens and keeps their whole rows in registers.
//
// Every product is computed transposed, C^T[feature, token] = W . X^T, with
// v_mfma_f32_16x16x32_bf16: 16 weight rows are the MFMA's A operand, the 16
// tokens its B operand and accumulator columns.  Lane l is token l % 16, group
// g = l / 16; an accumulator holds rows 4 g .. 4 g + 3.  The two MFMAs b = 0, 1
// of a 32-feature block take feature 8 (r / 4) + 4 b + r % 4 as row r, so a lane
// ends with the eight consecutive features 8 g .. 8 g + 7 of the block -- the
// B operand of the next product.  A product's bf16 output thus feeds the next
// one from the registers it was written to, and bias, residual, GELU and
// LayerNorm work on whole lanes; only two merges of the LayerNorm's tree and
// two levels of the softmax's sums cross lanes.
//
// The operation order is the wide path's: each product accumulates K in
// order, y = bf16(acc + bias) at the nn.Linear boundary, residual and GELU on
// those bf16 values, torch's Welford tree in the LayerNorm; the outputs are
// bit for bit the separate launches'.
//
// A row held by a lane: u32x4 x[D / 32], x[c] = the eight bf16 features
// 32 c + 8 g .. + 7 of the lane's token.
#pragma once

#include "common.h"
#include "welford.h"

namespace enc {
namespace narrow {

// The exact GELU's compact table: two slices of 231 16-byte chunks, copied to
// LDS by the workgroup.
constexpr int kGeluChunks = 231;                  // 16-byte chunks per sign, 1842 entries and 6 more
constexpr int kGeluSliceBytes = kGeluChunks * 16;
static_assert((kGeluHi - kGeluLo + 1) * 2 <= kGeluSliceBytes && (kGeluLo * 2) % 16 == 0, "table slices");

__device__ __forceinline__ bf16x8 as_frag(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }
__device__ __forceinline__ f32x4 zero4() { return f32x4{0.f, 0.f, 0.f, 0.f}; }

// LDS holds every MFMA operand as fragments of 1 KiB: the 16 bytes of lane l
// (row l % 16 of 16, eight values of K from 8 (l / 16)) at 16 l.  A fragment
// read is then one conflict-free 16-byte read per lane at a constant offset
// from 16 l, whatever the operand.
constexpr int kFrag = 512;  // bf16 elements
__device__ __forceinline__ bf16x8 lds_frag(const bf16_t* frags, int index, int lane) {
  return *reinterpret_cast<const bf16x8*>(frags + index * kFrag + lane * 8);
}
__device__ __forceinline__ u32x4 load16(const bf16_t* p) { return *reinterpret_cast<const u32x4*>(p); }

// The values of lanes l and l ^ 16 (l ^ 32), in the same order in both lanes.
struct Pair {
  float a, b;
};
__device__ __forceinline__ Pair across16(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}
__device__ __forceinline__ Pair across32(float v) {
  const uint32_t u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}

// Eight bf16 values of a u32x4 as floats
__device__ __forceinline__ void unpack8(u32x4 w, float (&v)[8]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[2 * e] = lo_bf16(w[e]);
    v[2 * e + 1] = hi_bf16(w[e]);
  }
}

// bf16(acc + bias) of a block's two accumulators (features 0..3 and 4..7)
__device__ __forceinline__ u32x4 bias_pack(const f32x4& a0, const f32x4& a1, u32x4 bias) {
  float b[8];
  unpack8(bias, b);
  return u32x4{pack_bf16x2(a0[0] + b[0], a0[1] + b[1]), pack_bf16x2(a0[2] + b[2], a0[3] + b[3]),
               pack_bf16x2(a1[0] + b[4], a1[1] + b[5]), pack_bf16x2(a1[2] + b[6], a1[3] + b[7])};
}
// bf16(x + bf16(acc + bias))
__device__ __forceinline__ u32x4 bias_residual(const f32x4& a0, const f32x4& a1, u32x4 bias, u32x4 x) {
  float b[8], r[8], y[8];
  unpack8(bias, b);
  unpack8(x, r);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    y[e] = r[e] + round_bf16(a0[e] + b[e]);
    y[4 + e] = r[4 + e] + round_bf16(a1[e] + b[4 + e]);
  }
  return u32x4{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]), pack_bf16x2(y[4], y[5]), pack_bf16x2(y[6], y[7])};
}

struct Stat {
  float mean, m2;
};
// Welford combine of two states of `count` elements each (a power of two):
// welford_merge_equal, which is symmetric in its operands.
__device__ __forceinline__ Stat stat_merge(Stat b, Stat a, float count) {
#pragma clang fp contract(off)
  const float delta = b.mean - a.mean;
  const float mean = 0.5f * a.mean + 0.5f * b.mean;
  const float m2 = __builtin_fmaf(delta * delta * count, 0.5f, a.m2 + b.m2);
  return {mean, m2};
}

// Statistics of the lane's row in packed_row_stats' order (welford.h): one
// state per 4-element vector, vector j = 8 c + 2 g + u (u = 0, 1), merged at
// distances D/8, .. 8 (registers), 4 and 2 (lane groups) and 1 (u).  The
// merges with empty states that torch's wider tree makes at the larger
// distances leave a state as it is, except that delta^2 * 0 is NaN once a
// vector's mean^2 overflows; that NaN is added at the end.
template <int D>
__device__ __forceinline__ void row_stats(const u32x4 (&x)[D / 32], float eps, float* mean, float* rstd) {
#pragma clang fp contract(off)
  constexpr int kC = D / 32;
  const float third = hw_rcp(3.f);
  Stat s[kC][2];
  float big = 0.f;
#pragma unroll
  for (int c = 0; c < kC; ++c) {
    float v[8];
    unpack8(x[c], v);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float m = v[4 * u] + 0.f, m2 = 0.f;
#pragma unroll
      for (int e = 1; e < 4; ++e) {
        const float delta = v[4 * u + e] - m;
        m = __builtin_fmaf(delta, e == 1 ? 0.5f : e == 2 ? third : 0.25f, m);
        const float p = delta * (v[4 * u + e] - m);
        m2 = e == 1 ? p : m2 + p;
      }
      s[c][u] = {m, m2};
      big = __builtin_elementwise_maximum(big, __builtin_fabsf(m));
    }
  }
  float count = 4.f;
#pragma unroll
  for (int step = kC / 2; step >= 1; step /= 2) {
#pragma unroll
    for (int c = 0; c < step; ++c)
#pragma unroll
      for (int u = 0; u < 2; ++u) s[c][u] = stat_merge(s[c][u], s[c + step][u], count);
    count *= 2.f;
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const Pair m = across32(s[0][u].mean), q = across32(s[0][u].m2);
    s[0][u] = stat_merge({m.a, q.a}, {m.b, q.b}, count);
  }
  count *= 2.f;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const Pair m = across16(s[0][u].mean), q = across16(s[0][u].m2);
    s[0][u] = stat_merge({m.a, q.a}, {m.b, q.b}, count);
  }
  count *= 2.f;
  const Stat t = stat_merge(s[0][0], s[0][1], count);
  const Pair b32 = across32(big);
  const Pair b16 = across16(__builtin_elementwise_maximum(b32.a, b32.b));
  big = __builtin_elementwise_maximum(b16.a, b16.b);
  *mean = t.mean;
  const float var = (t.m2 + (big * big) * 0.f) / static_cast<float>(D);
  *rstd = rsqrtf(var + eps);
}

// y = LayerNorm(x) of the lane's row
template <int D>
__device__ __forceinline__ void row_norm(const u32x4 (&x)[D / 32], const bf16_t* gamma, const bf16_t* beta, float eps,
                                         int g8, u32x4 (&y)[D / 32]) {
  float mean, rstd;
  row_stats<D>(x, eps, &mean, &rstd);
#pragma unroll
  for (int c = 0; c < D / 32; ++c) {
    float v[8], g[8], b[8], o[8];
    unpack8(x[c], v);
    unpack8(load16(gamma + 32 * c + g8), g);
    unpack8(load16(beta + 32 * c + g8), b);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = fmaf(g[e], rstd * (v[e] - mean), b[e]);
    y[c] = u32x4{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]), pack_bf16x2(o[4], o[5]), pack_bf16x2(o[6], o[7])};
  }
}

// GELU of eight bf16 values: through the table in LDS (tab: two slices of
// kGeluSliceBytes, magnitudes from kGeluLo; common.h's rules outside it) or, with
// no table, the erf.  (As gelu8_lds in gemm.hip; one function for both cost these
// kernels, at the edge of their registers, 1 to 3% in small batches.)
__device__ __forceinline__ u32x4 gelu8(u32x4 w, const char* tab, bool table) {
  if (table) {
    uint32_t u[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      u[2 * e] = w[e] & 0xffffu;
      u[2 * e + 1] = w[e] >> 16;
    }
    bool in_range = true;
#pragma unroll
    for (int e = 0; e < 8; ++e) in_range = in_range && (u[e] & 0x7fffu) - kGeluLo <= kGeluHi - kGeluLo;
    uint32_t g[8];
    if (__builtin_amdgcn_ballot_w64(!in_range) == 0) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        g[e] = *reinterpret_cast<const uint16_t*>(tab + (u[e] >> 15) * kGeluSliceBytes + ((u[e] & 0x7fffu) - kGeluLo) * 2);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t a = u[e] & 0x7fffu, s = u[e] >> 15;
        const uint32_t c = min(max(a, kGeluLo), kGeluHi);
        const uint32_t t = *reinterpret_cast<const uint16_t*>(tab + s * kGeluSliceBytes + (c - kGeluLo) * 2);
        const uint32_t half = f32_to_bf16(__uint_as_float(u[e] << 16) * 0.5f);
        const uint32_t big = (a + s > 0x7f80u) ? 0x7fc0u : (s != 0u ? 0x8000u : u[e]);
        g[e] = a < kGeluLo ? half : (a > kGeluHi ? big : t);
      }
    }
    return u32x4{g[0] | (g[1] << 16), g[2] | (g[3] << 16), g[4] | (g[5] << 16), g[6] | (g[7] << 16)};
  }
  float v[8];
  unpack8(w, v);
#pragma unroll 1
  for (int e = 0; e < 4; ++e) {  // (rolled: this path runs only before the table is filled)
    const float a = gelu_erf(v[0]), b = gelu_erf(v[1]);
#pragma unroll
    for (int k = 0; k < 6; ++k) v[k] = v[k + 2];
    v[6] = a;
    v[7] = b;
  }
  return u32x4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
}

// Copies the table's two slices to LDS (2 * kGeluChunks 16-byte chunks, 8 KiB
// written), by `waves` wavefronts.
__device__ __forceinline__ void gelu_to_lds(bf16_t* dst, const uint16_t* table, int wave, int waves, int lane) {
  const i32x4 rsrc = buffer_rsrc(table);
  for (int j = wave; j * 64 < 2 * kGeluChunks; j += waves) {
    const int q = min(64 * j + lane, 2 * kGeluChunks - 1);  // past the second slice: its last chunk again
    const int entry = q < kGeluChunks ? static_cast<int>(kGeluLo) + 8 * q
                                      : 0x8000 + static_cast<int>(kGeluLo) + 8 * (q - kGeluChunks);
    enc_buffer_load_lds(rsrc, lds_ptr(dst + j * 512), 16, entry * 2, 0, 0, 0);
  }
}

}  // namespace narrow
}  // namespace enc
