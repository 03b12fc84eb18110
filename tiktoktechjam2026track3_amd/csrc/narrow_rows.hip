// The two row-wise halves of a narrow model's layer (d_model and ffn_dim of
// 32, 64 or 128) around an attention launch of its own (sequences of more
// than 128 tokens, or batches that one launch would not serve faster):
//   narrow_qkv_kernel   norm1 and the packed QKV projection;
//   narrow_tail_kernel  out_proj + residual, norm2, the FFN + residual and,
//                       after the last layer, the final norm (many tokens;
//                       few take block_tail.hip's kernel).
// A wavefront owns 16 tokens whose rows stay in its registers (narrow.h); the
// weights are copied to LDS once per workgroup, as MFMA fragments, and the
// wavefronts then walk their slabs of 16 tokens without meeting again.
#include "kernels.h"
#include "narrow.h"

namespace enc {

namespace {

using namespace narrow;

// Copies `blocks` 32-row blocks of a [*, K] weight, from row0, to LDS:
// fragment (block, K step ks, b) at index (block * K / 32 + ks) * 2 + b.
template <int K>
__device__ __forceinline__ void weight_to_lds(bf16_t* dst, const bf16_t* weight, int row0, int blocks, int wave,
                                              int waves, int lane) {
  constexpr int kPer = K / 16;  // fragments of a block
  const i32x4 rsrc = buffer_rsrc(weight);
  const int l16 = lane & 15;
  const int voff = ((8 * (l16 >> 2) + (l16 & 3)) * K + 8 * (lane >> 4)) * 2;
  for (int f = wave; f < blocks * kPer; f += waves) {
    const int blk = f / kPer, ks = f % kPer / 2, b = f % 2;
    enc_buffer_load_lds(rsrc, lds_ptr(dst + f * kFrag), 16, voff, ((row0 + 32 * blk + 4 * b) * K + 32 * ks) * 2, 0, 0);
  }
}
// Copies a vector of len bf16 values (a multiple of 8, at most 512) to LDS.
__device__ __forceinline__ void vector_to_lds(bf16_t* dst, const bf16_t* src, int len, int lane) {
  if (lane * 8 < len) enc_buffer_load_lds(buffer_rsrc(src), lds_ptr(dst), 16, lane * 16, 0, 0, 0);
}

// One 32-feature block of a transposed product: K / 16 fragments, the lane's row.
template <int K>
__device__ __forceinline__ void block_product(const bf16_t* frags, int lane, const u32x4 (&x)[K / 32], f32x4& a0,
                                              f32x4& a1) {
  a0 = zero4();
  a1 = zero4();
#pragma unroll
  for (int ks = 0; ks < K / 32; ++ks) {
    a0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lds_frag(frags, 2 * ks, lane), as_frag(x[ks]), a0, 0, 0, 0);
    a1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lds_frag(frags, 2 * ks + 1, lane), as_frag(x[ks]), a1, 0, 0, 0);
  }
}

struct QkvArgs {
  const bf16_t *x, *gamma, *beta, *w, *bias;
  bf16_t *q, *k, *v_t;
  int S, hd_log2, ld_vt;
  int slabs, slabs_per_seq;
  int blocks;  // 32-feature blocks of [Q; K; V] per workgroup (blockIdx.y selects them)
  float eps;
};

template <int D>
constexpr int qkv_lds_bytes(int blocks) {
  return blocks * (D / 16) * kFrag * 2 + (2 * D + 32 * blocks) * 2;
}

// What bounds it: with many tokens the writes (64 x 1024 tokens of d_model 128,
// 67 MB in 19.4 us, 3.5 TB/s; norm and product as launches of their own took 38
// us); with few, latency, which splitting the feature blocks among workgroups
// shortens (launch_qkv).  16 wavefronts of at most 128 registers share one copy
// of the weights (96 KiB at d_model 128), four per SIMD.
template <int D>
__global__ void __launch_bounds__(1024) narrow_qkv_kernel(const QkvArgs a) {
  constexpr int kNB = D / 32, kBF = D / 16;
  extern __shared__ __attribute__((aligned(16))) bf16_t rows_lds[];
  bf16_t* frags = rows_lds;
  bf16_t* gamma = frags + a.blocks * kBF * kFrag;
  bf16_t* beta = gamma + D;
  bf16_t* bias = beta + D;

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int waves = blockDim.x / kWave;
  const int l16 = lane & 15;
  const int g = lane >> 4;
  const int g8 = 8 * g;
  const int first = blockIdx.y * a.blocks;

  weight_to_lds<D>(frags, a.w, 32 * first, a.blocks, wave, waves, lane);
  const int last_wave = waves - 1;
  if (wave == 0) vector_to_lds(gamma, a.gamma, D, lane);
  if (wave == min(1, last_wave)) vector_to_lds(beta, a.beta, D, lane);
  if (wave == min(2, last_wave)) vector_to_lds(bias, a.bias + 32 * first, 32 * a.blocks, lane);

  const int hd = 1 << a.hd_log2;
  auto load_rows = [&](int slab, u32x4 (&x)[kNB]) __attribute__((always_inline)) {
    const int seq = slab / a.slabs_per_seq;
    const int s = (slab - seq * a.slabs_per_seq) * 16 + l16;
    const bool valid = slab < a.slabs && s < a.S;
    const bf16_t* row = a.x + (static_cast<int64_t>(seq) * a.S + s) * D + g8;
#pragma unroll
    for (int c = 0; c < kNB; ++c) {
      x[c] = u32x4{0u, 0u, 0u, 0u};
      if (valid) x[c] = load16(row + 32 * c);
    }
  };
  int slab = blockIdx.x * waves + wave;
  u32x4 x[kNB];
  load_rows(slab, x);
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
  __syncthreads();

  while (slab < a.slabs) {
    u32x4 h[kNB];
    row_norm<D>(x, gamma, beta, a.eps, g8, h);
    const int seq = slab / a.slabs_per_seq;
    const int s0 = (slab - seq * a.slabs_per_seq) * 16;
    slab += gridDim.x * waves;
    if (slab < a.slabs) load_rows(slab, x);  // on their way during the products
    const int s = s0 + l16;
    const int64_t seq_off = static_cast<int64_t>(seq) * D * a.S;
#pragma unroll 1
    for (int i = 0; i < a.blocks; ++i) {
      const int which = (first + i) / kNB, c = (first + i) % kNB;
      const bf16_t* fr = frags + i * kBF * kFrag;
      if (which < 2) {
        f32x4 a0, a1;
        block_product<D>(fr, lane, h, a0, a1);
        const u32x4 y = bias_pack(a0, a1, load16(bias + 32 * i + g8));
        const int f = 32 * c + g8;
        if (s < a.S)
          *reinterpret_cast<u32x4*>((which == 0 ? a.q : a.k) + seq_off +
                                    (((f >> a.hd_log2) * a.S + s) << a.hd_log2) + (f & (hd - 1))) = y;
      } else {
        // V: the tokens are the A operand, so a lane holds the tokens 4 g ..
        // 4 g + 3 of one channel, eight bytes of its V^T row.  (The row's
        // stride is a multiple of 8: the padding columns are inside it.)
        f32x4 acc[2] = {zero4(), zero4()};
#pragma unroll
        for (int ks = 0; ks < kNB; ++ks) {
#pragma unroll
          for (int b = 0; b < 2; ++b)
            acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(h[ks]), lds_frag(fr, 2 * ks + b, lane), acc[b],
                                                             0, 0, 0);
        }
        const int row = 8 * (l16 >> 2) + (l16 & 3);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const float bb = bf16_to_f32(bias[32 * i + row + 4 * b]);
          if (s0 + 4 * g < a.ld_vt)
            *reinterpret_cast<u32x2*>(a.v_t + (static_cast<int64_t>(seq) * D + 32 * c + row + 4 * b) * a.ld_vt + s0 +
                                      4 * g) =
                u32x2{pack_bf16x2(acc[b][0] + bb, acc[b][1] + bb), pack_bf16x2(acc[b][2] + bb, acc[b][3] + bb)};
        }
      }
    }
  }
}

struct TailArgs {
  const bf16_t *ctx, *x;
  const bf16_t *wo, *bo, *g2, *be2, *w1, *b1, *w2, *b2;
  const bf16_t *final_g, *final_b;  // final norm, or null
  bf16_t* out;
  const uint8_t* row_mask;
  const uint16_t* gelu_table;
  const uint32_t* gelu_ready;
  int rows;
  float eps;
};

template <int D, int F>
struct Tail {
  static constexpr int kWo = 0, kW1 = D * D, kW2 = kW1 + D * F, kGelu = kW2 + D * F, kVecs = kGelu + 4096;
  static constexpr int kBo = kVecs, kG2 = kBo + D, kBe2 = kG2 + D, kB2 = kBe2 + D, kFg = kB2 + D, kFb = kFg + D,
                       kB1 = kFb + D;
  static constexpr int kLds = 2 * (kB1 + F);  // bytes
};

// What bounds it: VALU work and its latency, the weights' copy before it (64 x
// 1024 tokens of d_model and ffn_dim 128: 29 us, of which the 50 MB in and out
// would take 10; the five launches this replaced, three products and two norms,
// took 64).
template <int D, int F>
__global__ void __launch_bounds__(1024) narrow_tail_kernel(const TailArgs a) {
  using T = Tail<D, F>;
  constexpr int kNB = D / 32, kFB = F / 32;
  extern __shared__ __attribute__((aligned(16))) bf16_t rows_lds[];
  bf16_t* lds = rows_lds;

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int waves = blockDim.x / kWave;
  const int l16 = lane & 15;
  const int g8 = 8 * (lane >> 4);

  // The GELU table's ready flag: one reading for the workgroup, before any
  // table word is read (a clear flag selects the erf, the same bits).
  uint32_t* flag = reinterpret_cast<uint32_t*>(lds + T::kFb);
  if (threadIdx.x == 0) *flag = __hip_atomic_load(a.gelu_ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  weight_to_lds<D>(lds + T::kWo, a.wo, 0, kNB, wave, waves, lane);
  weight_to_lds<D>(lds + T::kW1, a.w1, 0, kFB, wave, waves, lane);
  weight_to_lds<F>(lds + T::kW2, a.w2, 0, kNB, wave, waves, lane);
  __syncthreads();
  const bool table = __builtin_amdgcn_readfirstlane(*flag) != 0;
  __syncthreads();
  if (table) gelu_to_lds(lds + T::kGelu, a.gelu_table, wave, waves, lane);
  for (int v = wave; v < 7; v += waves) {
    const bf16_t* src = v == 0 ? a.bo : v == 1 ? a.g2 : v == 2 ? a.be2 : v == 3 ? a.b2 : v == 4 ? a.final_g
                        : v == 5 ? a.final_b : a.b1;
    if (src != nullptr) vector_to_lds(lds + T::kBo + v * D, src, v == 6 ? F : D, lane);
  }

  const int slabs = (a.rows + 15) / 16;
  auto load_rows = [&](const bf16_t* src, int slab, u32x4 (&v)[kNB]) __attribute__((always_inline)) {
    const int r = slab * 16 + l16;
    const bf16_t* row = src + static_cast<int64_t>(r) * D + g8;
#pragma unroll
    for (int c = 0; c < kNB; ++c) {
      v[c] = u32x4{0u, 0u, 0u, 0u};
      if (r < a.rows) v[c] = load16(row + 32 * c);
    }
  };
  int slab = blockIdx.x * waves + wave;
  u32x4 x[kNB], h[kNB];  // h: the context, norm2's output, the final norm's
  load_rows(a.ctx, slab, h);
  load_rows(a.x, slab, x);
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
  __syncthreads();

  for (; slab < slabs; slab += gridDim.x * waves) {
    // (the vectors are read where they are used: hoisted out of this loop by
    // the compiler they spilled 61 registers, 39.6 us at the size above)
    asm volatile("" ::: "memory");
    const int r = slab * 16 + l16;
    const bool valid = r < a.rows;
    const bool keep = a.row_mask == nullptr || (valid && a.row_mask[r] != 0);
    // ---- out_proj + residual (rows masked out keep x) ----
#pragma unroll
    for (int c = 0; c < kNB; ++c) {
      f32x4 a0, a1;
      block_product<D>(lds + T::kWo + c * 32 * D, lane, h, a0, a1);
      const u32x4 y = bias_residual(a0, a1, load16(lds + T::kBo + 32 * c + g8), x[c]);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[c][e] = keep ? y[e] : x[c][e];
    }
    // ---- norm2, then the FFN + residual (rows masked out become 0): its
    // second product's K runs over the hidden features in order, so each 32
    // hidden features are consumed as they are produced ----
    row_norm<D>(x, lds + T::kG2, lds + T::kBe2, a.eps, g8, h);
    f32x4 o[kNB][2];
#pragma unroll
    for (int c = 0; c < kNB; ++c) {
      o[c][0] = zero4();
      o[c][1] = zero4();
    }
#pragma unroll 1
    for (int f = 0; f < kFB; ++f) {
      f32x4 a0, a1;
      block_product<D>(lds + T::kW1 + f * 32 * D, lane, h, a0, a1);
      const bf16x8 hf = as_frag(gelu8(bias_pack(a0, a1, load16(lds + T::kB1 + 32 * f + g8)),
                                      reinterpret_cast<const char*>(lds + T::kGelu), table));
#pragma unroll
      for (int c = 0; c < kNB; ++c) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
          o[c][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lds_frag(lds + T::kW2, (c * kFB + f) * 2 + b, lane), hf,
                                                            o[c][b], 0, 0, 0);
      }
    }
#pragma unroll
    for (int c = 0; c < kNB; ++c) {
      const u32x4 y = bias_residual(o[c][0], o[c][1], load16(lds + T::kB2 + 32 * c + g8), x[c]);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[c][e] = keep ? y[e] : 0u;
    }
    if (a.final_g != nullptr) {
      row_norm<D>(x, lds + T::kFg, lds + T::kFb, a.eps, g8, h);
#pragma unroll
      for (int c = 0; c < kNB; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[c][e] = keep ? h[c][e] : 0u;
    }
    if (valid) {
#pragma unroll
      for (int c = 0; c < kNB; ++c) *reinterpret_cast<u32x4*>(a.out + static_cast<int64_t>(r) * D + 32 * c + g8) = x[c];
    }
    load_rows(a.ctx, slab + gridDim.x * waves, h);
    load_rows(a.x, slab + gridDim.x * waves, x);
  }
}

// Wavefronts per workgroup for `slabs` slabs of 16 tokens: few enough that
// every CU gets a workgroup, 16 (four per SIMD) where there is work for them.
int waves_for(int64_t slabs, int cus) {
  int waves = 4;
  while (waves < 16 && static_cast<int64_t>(waves) * cus < slabs) waves *= 2;
  return waves;
}

template <typename K>
hipError_t allow_lds(K kernel, int bytes) {
  // above 64 KiB of dynamic LDS a kernel has to opt in
  if (bytes <= 64 * 1024) return hipSuccess;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

template <int D>
hipError_t launch_qkv(const QkvArgs& args, int cus, hipStream_t st) {
  static const hipError_t attr = allow_lds(narrow_qkv_kernel<D>, qkv_lds_bytes<D>(3 * D / 32));
  if (attr != hipSuccess) return attr;
  QkvArgs a = args;
  const int waves = waves_for(a.slabs, cus);
  const int groups = (a.slabs + waves - 1) / waves;
  constexpr int kBlocks = 3 * D / 32;
  a.blocks = kBlocks;
  const int grid = groups < cus ? groups : cus;
  // Few tokens: the 32-feature blocks are split among workgroups, which each
  // repeat the norm, as far as every CU still has at most one: a workgroup then
  // copies fewer weights and runs fewer products one after the other.  Four
  // layers of d_model 128, one workgroup for all blocks / split: 1 x 128 tokens
  // 90.2 / 71.7 us, 4 x 1024 261 / 245, 16 x 512 192 / 182.
  for (int split : {12, 6, 4, 3, 2}) {
    if (kBlocks % split == 0 && grid * split <= cus) {
      a.blocks = kBlocks / split;
      break;
    }
  }
  hipLaunchKernelGGL(narrow_qkv_kernel<D>, dim3(grid, kBlocks / a.blocks), dim3(waves * kWave),
                     qkv_lds_bytes<D>(a.blocks), st, a);
  return hipGetLastError();
}

template <int D, int F>
hipError_t launch_tail(const TailArgs& a, int cus, hipStream_t st) {
  static const hipError_t attr = allow_lds(narrow_tail_kernel<D, F>, Tail<D, F>::kLds);
  if (attr != hipSuccess) return attr;
  const int slabs = (a.rows + 15) / 16;
  const int waves = waves_for(slabs, cus);
  const int groups = (slabs + waves - 1) / waves;
  hipLaunchKernelGGL((narrow_tail_kernel<D, F>), dim3(groups < cus ? groups : cus), dim3(waves * kWave),
                     (Tail<D, F>::kLds), st, a);
  return hipGetLastError();
}

template <int D>
hipError_t launch_tail_f(int64_t f, const TailArgs& a, int cus, hipStream_t st) {
  switch (f) {
    case 32: return launch_tail<D, 32>(a, cus, st);
    case 64: return launch_tail<D, 64>(a, cus, st);
    case 128: return launch_tail<D, 128>(a, cus, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

bool narrow_rows_supported(int64_t rows, int64_t seq_len, int64_t d_model, int64_t heads, int64_t ffn_dim) {
  auto narrow = [](int64_t v) { return v == 32 || v == 64 || v == 128; };
  const int64_t hd = d_model / heads;
  return narrow(d_model) && narrow(ffn_dim) && d_model % heads == 0 && hd >= 8 && (hd & (hd - 1)) == 0 &&
         rows < (int64_t(1) << 31) - (int64_t(1) << 20) && seq_len <= (int64_t(1) << 23);
}

// The kernel pads every sequence to 16 tokens.  Even for one token that costs
// less than the LayerNorm launch it saves, except at d_model 128, whose products
// take twice d 64's time a slab, past about a thousand tokens (two layers, us,
// this / the two launches: d 128 1024 x 1 65.4 / 62.0, 65536 x 1 2116 / 2001,
// 16384 x 2 573 / 561, 16384 x 3 588 / 587, 64 x 1 37.0 / 41.2; d 64 1024 x 1 43.8 /
// 54.7, 8192 x 1 186 / 189).
bool narrow_qkv_faster(int64_t rows, int64_t seq_len, int64_t d_model) {
  return d_model < 128 || seq_len > 2 || rows < 1024;
}

hipError_t narrow_qkv_bf16(const bf16_t* x, const bf16_t* gamma, const bf16_t* beta, const bf16_t* w,
                           const bf16_t* bias, bf16_t* q, bf16_t* k, bf16_t* v_t, int64_t batch, int64_t seq_len,
                           int64_t d_model, int64_t heads, float eps, int cus, hipStream_t st) {
  if (!narrow_rows_supported(batch * seq_len, seq_len, d_model, heads, d_model)) return hipErrorInvalidValue;
  QkvArgs a{};
  a.x = x;
  a.gamma = gamma;
  a.beta = beta;
  a.w = w;
  a.bias = bias;
  a.q = q;
  a.k = k;
  a.v_t = v_t;
  a.S = static_cast<int>(seq_len);
  a.ld_vt = static_cast<int>(vt_stride(seq_len));
  for (int64_t hd = d_model / heads; hd > 1; hd /= 2) ++a.hd_log2;
  a.slabs_per_seq = static_cast<int>((seq_len + 15) / 16);
  const int64_t slabs = batch * a.slabs_per_seq;
  if (slabs >= (int64_t(1) << 31) - 65536) return hipErrorInvalidValue;
  a.slabs = static_cast<int>(slabs);
  a.eps = eps;
  switch (d_model) {
    case 32: return launch_qkv<32>(a, cus, st);
    case 64: return launch_qkv<64>(a, cus, st);
    default: return launch_qkv<128>(a, cus, st);
  }
}

// Few tokens: block_tail.hip splits each product's columns among the wavefronts
// of a 16-row slab, several times shorter from a slab's first load to its
// store; many: 16 slabs at once per CU.  Four layers with their attention, us
// (narrow_tail / block_tail): d_model 128 8 x 1000 286 / 278, 12 x 1024 293 /
// 297, 32 x 1024 449 / 495, 128 x 256 239 / 284; d_model 64 4 x 1024 235 / 231,
// 12 x 1024 242 / 254, 128 x 256 139 / 193; d_model 32 4 x 1024 230 / 227, 16 x
// 1024 231 / 253.
bool narrow_tail_faster(int64_t rows) { return rows > 8192; }

hipError_t narrow_tail_bf16(const BlockTailArgs& t, int64_t rows, int64_t d_model, int64_t ffn_dim, float eps, int cus,
                            hipStream_t st) {
  if (!narrow_rows_supported(rows, 1, d_model, 1, ffn_dim)) return hipErrorInvalidValue;
  TailArgs a{};
  const hipError_t e = gemm_gelu_table(st, &a.gelu_table, &a.gelu_ready);
  if (e != hipSuccess) return e;
  a.ctx = t.ctx;
  a.x = t.x;
  a.wo = t.wo;
  a.bo = t.bo;
  a.g2 = t.g2;
  a.be2 = t.be2;
  a.w1 = t.w1;
  a.b1 = t.b1;
  a.w2 = t.w2;
  a.b2 = t.b2;
  a.final_g = t.final_g;
  a.final_b = t.final_b;
  a.out = t.out;
  a.row_mask = t.row_mask;
  a.rows = static_cast<int>(rows);
  a.eps = eps;
  switch (d_model) {
    case 32: return launch_tail_f<32>(ffn_dim, a, cus, st);
    case 64: return launch_tail_f<64>(ffn_dim, a, cus, st);
    default: return launch_tail_f<128>(ffn_dim, a, cus, st);
  }
}

}  // namespace enc
