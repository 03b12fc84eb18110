// Fused block tail for narrow encoders (d_model and ffn_dim of 32, 64 or 128).
//
// After the attention, the reference's block runs (models.py:733-737)
//   x_attn = x + out_proj(context)          rows masked out keep x
//   h      = gelu(ffn_in(norm2(x_attn)))
//   x_out  = x_attn + ffn_out(h)            rows masked out become 0
// which the wide path launches as four kernels with [T, D] / [T, F] round
// trips through memory.  With d_model and ffn_dim <= 128 the three weight
// matrices fit in LDS together (104 KB at 128 / 128), so one persistent
// workgroup per CU loads them once and walks 16-row slabs of the tokens: the
// context and residual rows come in, every intermediate stays in LDS, and
// only x_out goes out (or, after the last layer, the final norm of it).  For
// these sizes the products are latency-bound: eight wavefronts take one
// 16-column block of each product, so a slab passes through three short chains
// (four wavefronts with two blocks each and 16-deep MFMAs, the biases loaded
// inside the chains: 9 us for 128 rows at 128 / 128 against 6).
//
// The arithmetic is the wide path's, operation for operation, so the output
// is bitwise the same: each product accumulates K sequentially in 32-deep
// MFMA steps (v_mfma_f32_16x16x32_bf16, the same bits as the 16-deep ones; the
// library splits none of these shapes), y = bf16(acc + bias) at the nn.Linear boundary, the
// residual adds and GELU-erf as in the GEMM epilogues, and norm2 through
// packed_row_stats, the LayerNorm kernel's reduction for rows of <= 128.
#include "common.h"
#include "kernels.h"
#include "welford.h"

namespace enc {

namespace {

constexpr int kTailRows = 16;       // rows per slab: the MFMA M dimension
constexpr int kTailWaves = 8;
constexpr int kTailThreads = kTailWaves * kWave;

// LDS row stride of a K-wide operand, bf16 elements: 16 bytes of padding put
// consecutive rows 4 banks apart, so the 16 rows of a fragment read spread
// over all 64 banks.
constexpr int tail_ld(int k) { return k + 8; }

// LDS layout, bf16 elements: Wo [D][D], W1 [F][D], W2 [D][F], then slab
// buffers A [16][D] (context, then norm2 output, then the block output), X
// [16][D] (residual, then x_attn) and Hd [16][F] (GELU output), each row
// padded to tail_ld.
constexpr size_t tail_lds_bytes(int d, int f) {
  return 2 * (static_cast<size_t>(d) * tail_ld(d) + static_cast<size_t>(f) * tail_ld(d) +
              static_cast<size_t>(d) * tail_ld(f) + kTailRows * (2 * static_cast<size_t>(tail_ld(d)) + tail_ld(f)));
}

// MFMA fragment of LDS row `row` (K-wide operand) at K offset k0: lane group g
// holds k0 + 8g .. k0 + 8g + 7 (A: row = l % 16; B: row = output column).
template <int K>
__device__ __forceinline__ bf16x8 tail_frag(const bf16_t* base, int row, int k0, int g) {
  return *reinterpret_cast<const bf16x8*>(base + row * tail_ld(K) + k0 + 8 * g);
}

// NROWS x K bf16 row-major (global) <-> registers <-> LDS (padded stride):
// chunk i of this thread is 16-byte chunk tid + kTailThreads i of the matrix.  The
// three weight matrices are loaded into registers together and only then
// stored, so their loads share one memory round trip.
template <int K, int NROWS>
struct TailRows {
  static constexpr int kChunks = K / 8;
  static constexpr int kTotal = NROWS * kChunks;
  static constexpr int kPer = (kTotal + kTailThreads - 1) / kTailThreads;  // chunks per thread
  __device__ static void load(u32x4 (&v)[kPer], const bf16_t* src, int tid) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = min(tid + i * kTailThreads, kTotal - 1);
      v[i] = *reinterpret_cast<const u32x4*>(src + static_cast<int64_t>(c / kChunks) * K + (c % kChunks) * 8);
    }
  }
  __device__ static void store(const u32x4 (&v)[kPer], bf16_t* dst, int tid) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = tid + i * kTailThreads;
      if (kTotal % kTailThreads == 0 || c < kTotal)
        *reinterpret_cast<u32x4*>(dst + (c / kChunks) * tail_ld(K) + (c % kChunks) * 8) = v[i];
    }
  }
};

template <int D, int F>
__global__ void __launch_bounds__(kTailThreads)
block_tail_kernel(const bf16_t* __restrict__ ctx, const bf16_t* __restrict__ x, const bf16_t* __restrict__ wo,
                  const bf16_t* __restrict__ bo, const bf16_t* __restrict__ g2, const bf16_t* __restrict__ be2,
                  const bf16_t* __restrict__ w1, const bf16_t* __restrict__ b1, const bf16_t* __restrict__ w2,
                  const bf16_t* __restrict__ b2, bf16_t* __restrict__ out, int rows, float eps,
                  const uint8_t* __restrict__ row_mask, const bf16_t* __restrict__ final_g,
                  const bf16_t* __restrict__ final_b) {
  static_assert((D == 32 || D == 64 || D == 128) && (F == 32 || F == 64 || F == 128), "d_model, ffn_dim");
  constexpr int kLdD = tail_ld(D), kLdF = tail_ld(F);
  constexpr int kSlabChunks = kTailRows * (D / 8);  // 16-byte chunks of a [16][D] slab
  static_assert(kSlabChunks <= kTailThreads, "one chunk of each slab operand per thread");
  static_assert(D / 16 <= kTailWaves && F / 16 <= kTailWaves, "one column block per wavefront");
  extern __shared__ __attribute__((aligned(16))) bf16_t tail_lds[];
  bf16_t* sWo = tail_lds;
  bf16_t* sW1 = sWo + D * kLdD;
  bf16_t* sW2 = sW1 + F * kLdD;
  bf16_t* sA = sW2 + D * kLdF;
  bf16_t* sX = sA + kTailRows * kLdD;
  bf16_t* sH = sX + kTailRows * kLdD;

  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int l16 = lane & 15;
  const int g = lane >> 4;

  // the slab's context and residual chunks travel in registers one slab ahead
  const int slabs = (rows + kTailRows - 1) / kTailRows;
  const int my_r = tid / (D / 8), my_ch = tid % (D / 8);
  const bool has_chunk = tid < kSlabChunks;
  u32x4 next_a = {0u, 0u, 0u, 0u}, next_x = {0u, 0u, 0u, 0u};
  auto fetch = [&](int slab) {
    next_a = u32x4{0u, 0u, 0u, 0u};
    next_x = u32x4{0u, 0u, 0u, 0u};
    const int r = slab * kTailRows + my_r;
    if (has_chunk && slab < slabs && r < rows) {
      next_a = *reinterpret_cast<const u32x4*>(ctx + static_cast<int64_t>(r) * D + my_ch * 8);
      next_x = *reinterpret_cast<const u32x4*>(x + static_cast<int64_t>(r) * D + my_ch * 8);
    }
  };
  fetch(blockIdx.x);

  // norm2's gamma / beta for this lane's vector (rows of D = 4 L elements)
  constexpr int L = D / 4;
  constexpr int R = kWave / L;  // rows per wavefront in the norm2 pass
  const int seg = lane / L, j = lane % L;
  const u32x2 gw = *reinterpret_cast<const u32x2*>(g2 + 4 * j);
  const u32x2 bw = *reinterpret_cast<const u32x2*>(be2 + 4 * j);
  // the final norm's (optional)
  const bool final_norm = final_g != nullptr;
  u32x2 gn = {0u, 0u}, bn = {0u, 0u};
  if (final_norm) {
    gn = *reinterpret_cast<const u32x2*>(final_g + 4 * j);
    bn = *reinterpret_cast<const u32x2*>(final_b + 4 * j);
  }
  // this lane's column of the three products and its biases (a wavefront
  // takes one 16-column block of each; past the width, the last column's)
  const int col = wave * 16 + l16;
  const float bias_o = bf16_to_f32(bo[min(col, D - 1)]);
  const float bias_1 = bf16_to_f32(b1[min(col, F - 1)]);
  const float bias_2 = bf16_to_f32(b2[min(col, D - 1)]);

  {
    using RWo = TailRows<D, D>;
    using RW1 = TailRows<D, F>;
    using RW2 = TailRows<F, D>;
    u32x4 vo[RWo::kPer], v1[RW1::kPer], v2[RW2::kPer];
    RWo::load(vo, wo, tid);
    RW1::load(v1, w1, tid);
    RW2::load(v2, w2, tid);
    RWo::store(vo, sWo, tid);
    RW1::store(v1, sW1, tid);
    RW2::store(v2, sW2, tid);
  }

  for (int slab = blockIdx.x; slab < slabs; slab += gridDim.x) {
    const int r0 = slab * kTailRows;
    __syncthreads();  // the previous slab's output copy has read sA (and the weights have landed)
    if (has_chunk) {
      *reinterpret_cast<u32x4*>(sA + my_r * kLdD + my_ch * 8) = next_a;
      *reinterpret_cast<u32x4*>(sX + my_r * kLdD + my_ch * 8) = next_x;
    }
    fetch(slab + gridDim.x);
    // Row-mask verdicts of this lane's output rows 4g .. 4g+3, taken before
    // the products: with no branch between an MFMA and the reads of its
    // result, the compiler's wait states before those reads stay in place
    // (a mask test between them left a result register read two
    // instructions after its MFMA, before the write landed).
    bool keep[4];
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int r = r0 + 4 * g + jj;
      keep[jj] = row_mask == nullptr || (r < rows && row_mask[r] != 0);
    }
    __syncthreads();

    // ---- out_proj + residual (rows masked out keep the residual) -> sX ----
    if (wave < D / 16) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < D / 32; ++ks)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tail_frag<D>(sA, l16, ks * 32, g),
                                                        tail_frag<D>(sWo, col, ks * 32, g), acc, 0, 0, 0);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const int r = 4 * g + jj;
        const float y = round_bf16(acc[jj] + bias_o);  // nn.Linear output boundary
        bf16_t* px = sX + r * kLdD + col;
        const bf16_t old = *px;
        *px = keep[jj] ? f32_to_bf16(bf16_to_f32(old) + y) : old;
      }
    }
    __syncthreads();

    // ---- norm2 (no row mask) -> sA ----
    for (int p = 0; p < kTailRows; p += kTailWaves * R) {
      const int r = p + wave * R + seg;
      const int rr = r < kTailRows ? r : kTailRows - 1;  // lanes past the slab only join the shuffles
      const u32x2 w = *reinterpret_cast<const u32x2*>(sX + rr * kLdD + 4 * j);
      const float v[4] = {lo_bf16(w[0]), hi_bf16(w[0]), lo_bf16(w[1]), hi_bf16(w[1])};
      float mean, rstd;
      packed_row_stats<L>(v, j, seg, eps, &mean, &rstd);
      if (r < kTailRows) {
        const float ga[4] = {lo_bf16(gw[0]), hi_bf16(gw[0]), lo_bf16(gw[1]), hi_bf16(gw[1])};
        const float be[4] = {lo_bf16(bw[0]), hi_bf16(bw[0]), lo_bf16(bw[1]), hi_bf16(bw[1])};
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = fmaf(ga[e], rstd * (v[e] - mean), be[e]);
        *reinterpret_cast<u32x2*>(sA + r * kLdD + 4 * j) = u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
      }
    }
    __syncthreads();

    // ---- ffn_in + GELU -> sH ----
    if (wave < F / 16) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < D / 32; ++ks)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tail_frag<D>(sA, l16, ks * 32, g),
                                                        tail_frag<D>(sW1, col, ks * 32, g), acc, 0, 0, 0);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const float y = round_bf16(acc[jj] + bias_1);
        sH[(4 * g + jj) * kLdF + col] = f32_to_bf16(gelu_erf(y));
      }
    }
    __syncthreads();

    // ---- ffn_out + residual (rows masked out become 0) -> sA ----
    if (wave < D / 16) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < F / 32; ++ks)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tail_frag<F>(sH, l16, ks * 32, g),
                                                        tail_frag<F>(sW2, col, ks * 32, g), acc, 0, 0, 0);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const int r = 4 * g + jj;
        const float y = round_bf16(acc[jj] + bias_2);
        sA[r * kLdD + col] = keep[jj] ? f32_to_bf16(bf16_to_f32(sX[r * kLdD + col]) + y) : bf16_t(0);
      }
    }
    __syncthreads();

    if (!final_norm) {
      // ---- block output, 16-byte stores ----
      if (has_chunk && r0 + my_r < rows)
        *reinterpret_cast<u32x4*>(out + static_cast<int64_t>(r0 + my_r) * D + my_ch * 8) =
            *reinterpret_cast<const u32x4*>(sA + my_r * kLdD + my_ch * 8);
    } else {
      // ---- the final norm of the block output rows (rows masked out stay 0) ----
      for (int p = 0; p < kTailRows; p += kTailWaves * R) {
        const int r = p + wave * R + seg;
        const int rr = r < kTailRows ? r : kTailRows - 1;  // lanes past the slab only join the shuffles
        const u32x2 w = *reinterpret_cast<const u32x2*>(sA + rr * kLdD + 4 * j);
        const float v[4] = {lo_bf16(w[0]), hi_bf16(w[0]), lo_bf16(w[1]), hi_bf16(w[1])};
        float mean, rstd;
        packed_row_stats<L>(v, j, seg, eps, &mean, &rstd);
        if (r < kTailRows && r0 + r < rows) {
          const bool live = row_mask == nullptr || row_mask[r0 + r] != 0;
          const float ga[4] = {lo_bf16(gn[0]), hi_bf16(gn[0]), lo_bf16(gn[1]), hi_bf16(gn[1])};
          const float be[4] = {lo_bf16(bn[0]), hi_bf16(bn[0]), lo_bf16(bn[1]), hi_bf16(bn[1])};
          float o[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = live ? fmaf(ga[e], rstd * (v[e] - mean), be[e]) : 0.f;
          *reinterpret_cast<u32x2*>(out + static_cast<int64_t>(r0 + r) * D + 4 * j) =
              u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
        }
      }
    }
  }
}

template <int D, int F>
hipError_t launch_tail(const BlockTailArgs& a, int rows, float eps, int num_cus, hipStream_t st) {
  auto kernel = block_tail_kernel<D, F>;
  constexpr size_t kLds = tail_lds_bytes(D, F);
  if constexpr (kLds > 64 * 1024) {
    // above 64 KiB of dynamic LDS the kernel has to opt in (once per process)
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       static_cast<int>(kLds));
    if (attr != hipSuccess) return attr;
  }
  const int slabs = (rows + kTailRows - 1) / kTailRows;
  const int grid = slabs < num_cus ? slabs : num_cus;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(kTailThreads), kLds, st, a.ctx, a.x, a.wo, a.bo, a.g2, a.be2, a.w1,
                     a.b1, a.w2, a.b2, a.out, rows, eps, a.row_mask, a.final_g, a.final_b);
  return hipGetLastError();
}

template <int D>
hipError_t launch_tail_f(int f, const BlockTailArgs& a, int rows, float eps, int num_cus, hipStream_t st) {
  switch (f) {
    case 32: return launch_tail<D, 32>(a, rows, eps, num_cus, st);
    case 64: return launch_tail<D, 64>(a, rows, eps, num_cus, st);
    case 128: return launch_tail<D, 128>(a, rows, eps, num_cus, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

bool block_tail_supported(int64_t d_model, int64_t ffn_dim) {
  auto ok = [](int64_t v) { return v == 32 || v == 64 || v == 128; };
  return ok(d_model) && ok(ffn_dim);
}

hipError_t block_tail_bf16(const BlockTailArgs& a, int64_t rows, int64_t d_model, int64_t ffn_dim, float eps,
                           int num_cus, hipStream_t stream) {
  if (rows == 0) return hipSuccess;
  if (!block_tail_supported(d_model, ffn_dim) || rows >= (int64_t(1) << 31)) return hipErrorInvalidValue;
  // the kernel reads x and writes out through restrict pointers
  if (a.out == a.x) return hipErrorInvalidValue;
  const int r = static_cast<int>(rows);
  switch (d_model) {
    case 32: return launch_tail_f<32>(static_cast<int>(ffn_dim), a, r, eps, num_cus, stream);
    case 64: return launch_tail_f<64>(static_cast<int>(ffn_dim), a, r, eps, num_cus, stream);
    case 128: return launch_tail_f<128>(static_cast<int>(ffn_dim), a, r, eps, num_cus, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace enc
