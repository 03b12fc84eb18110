// The whole encoder forward of a narrow model (d_model and ffn_dim of 32, 64
// or 128) over sequences of at most 128 tokens, in one launch.
//
// A sequence of S tokens is ceil(S / 16) wavefronts of 16 tokens; a workgroup
// of eight wavefronts holds up to four sequences and runs every layer on them:
// the tokens' rows stay in registers from the first norm to the last
// (narrow.h), K and V^T go through LDS (the only exchange between
// wavefronts), and the weights stream from L2 through an LDS ring that the
// eight wavefronts share.  Activations are read once and written once.
#include "kernels.h"
#include "narrow.h"

namespace enc {

namespace {

using namespace narrow;

constexpr float kMinFastGap = -69.0f;  // below it the corrected quotient is not used (attention_exact.h)
constexpr int kWaves = 8;

struct NarrowArgs {
  const bf16_t* x;
  bf16_t* out;
  const int32_t* kv_len;
  const uint8_t* key_mask;
  const uint8_t* row_mask;
  const bf16_t* final_g;  // final norm, or null
  const bf16_t* final_b;
  const uint16_t* gelu_table;
  const uint32_t* gelu_ready;
  int B, S, F, layers, causal;
  float eps, scale;
  const bf16_t* w[kNarrowMaxLayers][12];
};

// Which keys this wavefront's queries see (uniform but for the lane's row).
struct Keys {
  int base;       // the sequence's first 32-key block in the workgroup's K and V^T
  int q32;        // the 32-token block of the queries
  int qoff;       // the lane's query in that block
  int blocks;     // 32-key blocks with a score to form
  int pv_blocks;  // ... and with values to add (whole 64-key tiles, as the attention kernel walks them)
  bool causal;
  bool zero_row;  // the lane's query is padding
  uint32_t valid[4];
};

// 16 queries of one head against up to four 32-key blocks, as
// attention_exact.h computes rows of at most 128 keys (same operations, same
// order): raw dots, their maximum, weights, the row sum's 64-lane order, the
// corrected division, P.V in key order.  Key 32 kb + 8 g + i is in s[kb][i].
//   qf: the head's queries; sK: K fragments, (2 kb + b) (GC / 32) + chunk, row r
//   of fragment b being key 8 (r / 4) + 4 b + r % 4 of the block; sV: V^T
//   fragments, kb (GC / 16) + 2 (32-channel block) + b, rows likewise channels
template <int GC, int HD>
__device__ __forceinline__ void head_attention(const bf16x8 (&qf)[HD < 32 ? 1 : HD / 32], const bf16_t* sK,
                                               const bf16_t* sV, int head, const Keys& keys, float scale, int lane,
                                               u32x4 (&ctx)[HD < 32 ? 1 : HD / 32]) {
  constexpr bool kPow2 = HD == 64;
  constexpr int kSteps = HD < 32 ? 1 : HD / 32;  // 32-channel steps of q.k, 32-channel blocks of the context
  const int g = lane >> 4;
  // Excluded keys: bit i of the lane's byte of the block's word allows the key
  // in register i; an excluded key's dot product becomes -inf (weight 0) and
  // counts as +inf in the minimum.  need[kb]: some lane may exclude a key.
  // (The bytes are made opaque here, per head: the compiler would otherwise
  // test all bits once per kernel and carry the verdicts through spills.)
  float s[4][8];
  bool need[4];
  float mx = -INFINITY, mn = INFINITY;
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const bool diag = keys.causal && kb == keys.q32;
    need[kb] = diag || keys.valid[kb] != 0xffffffffu;
    if (kb >= keys.blocks) {
#pragma unroll
      for (int i = 0; i < 8; ++i) s[kb][i] = 0.f;
      continue;
    }
    f32x4 d0 = zero4(), d1 = zero4();
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks) {
      const int chunk = HD < 32 ? head / 4 : head * (HD / 32) + ks;
      bf16x8 k0 = lds_frag(sK, (2 * (keys.base + kb)) * (GC / 32) + chunk, lane);
      bf16x8 k1 = lds_frag(sK, (2 * (keys.base + kb) + 1) * (GC / 32) + chunk, lane);
      if (HD < 32) {  // four heads share a chunk: the other three's channels as zeros
        const u32x4 none = {0u, 0u, 0u, 0u};
        k0 = g == (head & 3) ? k0 : as_frag(none);
        k1 = g == (head & 3) ? k1 : as_frag(none);
      }
      d0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, qf[ks], d0, 0, 0, 0);
      d1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1, qf[ks], d1, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[kb][i] = d0[i];
      s[kb][4 + i] = d1[i];
    }
    if (need[kb]) {
      uint32_t byte = (diag ? keys.valid[kb] & (0xffffffffu >> (31 - keys.qoff)) : keys.valid[kb]) >> (8 * g);
      asm("" : "+v"(byte));
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t on = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(byte), i, 1));
        const uint32_t v = __float_as_uint(s[kb][i]);
        mn = __builtin_elementwise_minimum(mn, __uint_as_float((v & on) | (0x7f800000u & ~on)));
        s[kb][i] = __uint_as_float((v & on) | (0xff800000u & ~on));
        mx = __builtin_elementwise_maximum(mx, s[kb][i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        mx = __builtin_elementwise_maximum(mx, __builtin_elementwise_maximum(s[kb][i], s[kb][i + 1]));
        mn = __builtin_elementwise_minimum(mn, __builtin_elementwise_minimum(s[kb][i], s[kb][i + 1]));
      }
    }
  }
  {
    const Pair a = across32(mx), b = across32(mn);
    const Pair c = across16(__builtin_elementwise_maximum(a.a, a.b)), d = across16(__builtin_elementwise_minimum(b.a, b.b));
    mx = __builtin_elementwise_maximum(c.a, c.b);
    mn = __builtin_elementwise_minimum(d.a, d.b);
  }
  const bool none = mx == -INFINITY;
  const float raw_max = none ? -INFINITY : round_bf16(mx);
  const float row_max = none ? -INFINITY : (kPow2 ? raw_max * scale : round_bf16(raw_max * scale));
  const float min_q = round_bf16(mn);
  const float row_min = kPow2 ? min_q * scale : round_bf16(min_q * scale);
  // (a NaN among the scores makes the row's sum NaN and its context zero
  // either way)
  const bool slow_div = __builtin_amdgcn_ballot_w64(mn != INFINITY && row_min - row_max < kMinFastGap) != 0;
  const ExpfScaled ec = expf_scaled_consts(scale);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    if (kb >= keys.blocks) continue;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float v = round_bf16(s[kb][i]);
      s[kb][i] = kPow2 ? v - raw_max : round_bf16(v * scale) - row_max;
    }
    if (need[kb] || slow_div) {
      // the clamped exponential: an excluded key's gap is -inf, its weight 0
#pragma unroll
      for (int i = 0; i < 8; ++i) s[kb][i] = kPow2 ? expf_nonpos_scaled(s[kb][i], ec) : expf_nonpos(s[kb][i]);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        s[kb][i] = kPow2 ? expf_nonpos_scaled_unclamped(s[kb][i], ec) : expf_nonpos_unclamped(s[kb][i]);
    }
  }
  // partial[key % 64] = e(key) + e(key + 64), then the 64-lane butterfly:
  // distance 32 (block parity), 16 and 8 (lane groups), 4, 2, 1 (registers).
  // A lane swap of two partials does both their sums at once: after it a lane
  // half (row of 16) holds the one or the other, and the last levels cross
  // lanes where the plain form would cross registers.
  float c[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) c[i] = (s[0][i] + s[2][i]) + (s[1][i] + s[3][i]);
  float d[4];  // lane half h: partial i + 4 h
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(c[i]), __float_as_uint(c[i + 4]), false, false);
    d[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  float e2[2];  // row parity p: partial i + 2 p + 4 h
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(d[i]), __float_as_uint(d[i + 2]), false, false);
    e2[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    const Pair four = across32(e2[i]);
    const Pair two = across16(four.a + four.b);
    e2[i] = two.a + two.b;
  }
  const float row_sum = e2[0] + e2[1];
  const float inv_sum = 1.0f / row_sum;

  f32x4 o[kSteps][2];
#pragma unroll
  for (int db = 0; db < kSteps; ++db) {
    o[db][0] = zero4();
    o[db][1] = zero4();
  }
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    if (kb >= keys.pv_blocks) continue;
    bf16x8 pf;
    if (!slow_div) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float e = s[kb][i];
        const float q = e * inv_sum;
        pf[i] = static_cast<__bf16>(fmaf(fmaf(-q, row_sum, e), inv_sum, q));
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) pf[i] = static_cast<__bf16>(s[kb][i] / row_sum);
    }
#pragma unroll
    for (int db = 0; db < kSteps; ++db) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        // (head dim 8: row r takes the head's channel 4 b + r % 4, so every
        // lane group ends with the head's eight channels)
        const int frag = (keys.base + kb) * (GC / 16) + 2 * (HD < 32 ? head / 4 : head * (HD / 32) + db) + b;
        const int at = HD < 32 ? 4 * (head & 3) + (lane & 3) + (lane & 48) : lane;
        o[db][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lds_frag(sV, frag, at), pf, o[db][b], 0, 0, 0);
      }
    }
  }
  const bool zero = keys.zero_row || !(row_sum > 0.f);
#pragma unroll
  for (int db = 0; db < kSteps; ++db) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const uint32_t w = pack_bf16x2(o[db][b][2 * e], o[db][b][2 * e + 1]);
        ctx[db][2 * b + e] = zero ? 0u : w;
      }
    }
  }
}

// Sizes of the kernel at (D, HD).  The weights of a layer are a sequence of
// stages of kSB 32-row blocks, in the order they are used:
//   per channel group: Q rows, K rows, V rows (kQS stages each); then
//   out_proj's rows; then per 32 kSB hidden features ffn_in's rows and
//   ffn_out's columns.
// The heads run in groups of kGC channels so that K and V^T of a group, the
// two stages, the GELU table and two layers' vectors fit twice in a CU's LDS.
// A stage is as long as that allows: each costs a barrier (32-row stages at
// d_model 128: 3.39 ms against 3.21 for four layers of 10000 sequences).
template <int D, int HD>
struct Narrow {
  static constexpr int kNB = D / 32;                         // 32-feature blocks (u32x4 per lane) of a row
  static constexpr int kBF = D / 16;                         // fragments of a 32-row block
  static constexpr int kGC = D == 128 && HD <= 64 ? 64 : D;  // channels per head group
  static constexpr int kNG = kGC / 32;
  static constexpr int kGroups = D / kGC;
  static constexpr int kSB = D == 32 ? 1 : 2;
  static constexpr int kQS = kNG / kSB;
  static constexpr int kStage = kSB * kBF * kFrag;           // elements
  static constexpr int kKV = 128 * kGC;                      // elements of K, and of V^T
  static constexpr int kVecs = 2560 / 2;                     // (9 D + F) bf16 at most, per layer
  static constexpr int kGelu = 4096;                         // GELU table, elements
  static constexpr int kLds = 2 * (2 * kKV + 2 * kStage + kGelu + 2 * kVecs);
};

// Offsets of a layer's vectors in its LDS block (elements)
template <int D>
struct Vecs {
  static constexpr int kQkv = 0, kOut = 3 * D, kG1 = 4 * D, kB1 = 5 * D, kG2 = 6 * D, kB2 = 7 * D, kFfnOut = 8 * D,
                       kFfnIn = 9 * D;
};

// Requests layer vector v (0 .. 7) into the block.
template <int D>
__device__ __forceinline__ void vec_to_lds(bf16_t* block, const bf16_t* const* w, int v, int F, int lane) {
  // qkv_proj.bias, out_proj.bias, norm1, norm2, ffn_out.bias, ffn_in.bias
  const int src = v == 0 ? 3 : v == 1 ? 5 : v == 2 ? 0 : v == 3 ? 1 : v == 4 ? 6 : v == 5 ? 7 : v == 6 ? 11 : 9;
  const int at = v == 0 ? 0 : (v + 2) * D;
  const int len = v == 0 ? 3 * D : v == 7 ? F : D;
  if (lane * 8 < len) enc_buffer_load_lds(buffer_rsrc(w[src]), lds_ptr(block + at), 16, lane * 16, 0, 0, 0);
}

// One 32-feature block of a transposed product: the block's fragments (2 per
// K step, one for each b), the lane's row.
template <int D>
__device__ __forceinline__ void block_product(const bf16_t* frags, int lane, const u32x4 (&x)[D / 32], f32x4& a0,
                                              f32x4& a1) {
  a0 = zero4();
  a1 = zero4();
#pragma unroll
  for (int ks = 0; ks < D / 32; ++ks) {
    a0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lds_frag(frags, 2 * ks, lane), as_frag(x[ks]), a0, 0, 0, 0);
    a1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lds_frag(frags, 2 * ks + 1, lane), as_frag(x[ks]), a1, 0, 0, 0);
  }
}

// What bounds it: VALU issue (rocprofv3 on 10000 sequences of 128 tokens, d_model
// 128, head dim 32: 79% of the cycles at four an instruction, 4857 instructions a
// wavefront and layer with 236 MFMAs, more than half of them the exact softmax);
// in a small batch the latency of one workgroup, 30 us a layer at 32 channels a
// head.  16 tokens a wavefront leave 128 registers, four wavefronts per SIMD (two
// workgroups of 77 KiB per CU; one at head dim 128), at the price of spills: 7 to
// 57 vector registers at d_model 128 and at head dim 8 of 64, 18 to 54 scalar
// ones, to vector lanes, everywhere.  32 tokens a wavefront at two per SIMD ran
// the four layers of that batch in 3.71 ms against 3.17 ms here, the launches
// this replaced (norm, QKV, attention, out_proj, norm, ffn_in, ffn_out a layer)
// in 7.30 ms.
template <int D, int HD>
__global__ void __launch_bounds__(kWaves * kWave, 4) narrow_forward_kernel(const NarrowArgs a) {
  using N = Narrow<D, HD>;
  using V = Vecs<D>;
  constexpr int kNB = N::kNB, kNG = N::kNG, kGC = N::kGC, kSB = N::kSB, kQS = N::kQS, kBF = N::kBF;
  extern __shared__ __attribute__((aligned(16))) bf16_t narrow_lds[];
  bf16_t* sK = narrow_lds;
  bf16_t* sV = sK + N::kKV;
  bf16_t* ring = sV + N::kKV;
  bf16_t* gelu = ring + 2 * N::kStage;
  bf16_t* vecs = gelu + N::kGelu;  // layer l's vectors in block l & 1

  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int l16 = lane & 15;
  const int g = lane >> 4;
  const int g8 = 8 * g;

  // this wavefront's sequence and 16-token block of it; a causal sequence's
  // later blocks have more keys, so odd workgroups hand the blocks out in
  // reverse
  const int S = a.S;
  const int nw = (S + 15) / 16, nk = (S + 31) / 32;
  const int spb = min(kWaves / nw, 4 / nk);
  const int in_group = wave / nw;
  int qb = wave - in_group * nw;
  if (blockIdx.x & 1) qb = nw - 1 - qb;
  const int seq = blockIdx.x * spb + in_group;
  const bool live = in_group < spb && seq < a.B;  // uniform per wavefront
  // A lane past the sequence repeats its last token, in every step and in the
  // output's store (the same bits to the same row): its value meets zero
  // weights only, and one that is not finite would still reach the context, as
  // zeros in the token's place would that run norm1's bias through each layer.
  const int s = min(16 * qb + l16, S - 1);
  const int64_t row = static_cast<int64_t>(seq) * S + s;

  Keys keys;
  keys.base = live ? in_group * nk : 0;
  keys.q32 = qb / 2;
  keys.qoff = 16 * (qb & 1) + l16;
  keys.causal = a.causal != 0;
  int kv_limit = S;
  if (a.kv_len != nullptr && live) kv_limit = min(S, max(0, a.kv_len[seq]));
  kv_limit = __builtin_amdgcn_readfirstlane(kv_limit);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const int left = kv_limit - 32 * kb;
    keys.valid[kb] = left >= 32 ? 0xffffffffu : left > 0 ? (1u << left) - 1u : 0u;
    if (a.key_mask != nullptr && live) {
      const int key = 32 * kb + (lane & 31);
      const bool on = key < S && a.key_mask[static_cast<int64_t>(seq) * S + key] != 0;
      keys.valid[kb] &= static_cast<uint32_t>(__builtin_amdgcn_ballot_w64(on));
    }
  }
  const int limit_blocks = min(nk, 2 * ((kv_limit + 63) / 64));
  keys.blocks = keys.causal ? min(limit_blocks, keys.q32 + 1) : limit_blocks;
  keys.pv_blocks = keys.causal ? min(limit_blocks, (keys.q32 | 1) + 1) : limit_blocks;
  const bool attends = live && !(a.kv_len != nullptr && 16 * qb >= kv_limit);
  keys.zero_row = a.kv_len != nullptr && s >= kv_limit;
  const bool keep = a.row_mask == nullptr || (live && a.row_mask[row] != 0);

  u32x4 x[kNB];
#pragma unroll
  for (int c = 0; c < kNB; ++c) {
    x[c] = u32x4{0u, 0u, 0u, 0u};
    if (live) x[c] = load16(a.x + row * D + 32 * c + g8);
  }
  // The GELU table's ready flag: one reading for the workgroup, before any
  // table word is read (a clear flag selects the erf, the same bits).  V^T's
  // slots of tokens that no wavefront owns (an odd number of 16-token blocks)
  // are read with zero weights: zeros, once.
  if (tid == 0)
    *reinterpret_cast<uint32_t*>(sK) = __hip_atomic_load(a.gelu_ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int i = tid; i < N::kKV / 8; i += kWaves * kWave) *reinterpret_cast<u32x4*>(sV + 8 * i) = u32x4{0u, 0u, 0u, 0u};
  __syncthreads();
  const bool table = __builtin_amdgcn_readfirstlane(*reinterpret_cast<const uint32_t*>(sK)) != 0;
  if (table) gelu_to_lds(gelu, a.gelu_table, wave, kWaves, lane);
  for (int v = wave; v < 8; v += kWaves) vec_to_lds<D>(vecs, a.w[0], v, a.F, lane);

  // The ring of two stages.  begin_stage waits for the current stage's
  // fragments and meets the other wavefronts; then, with the stage's MFMAs on
  // their way, the next stage is requested into the slot that everyone has
  // left.  Fragment f of a stage of rows is (block f / kBF, K step f % kBF / 2,
  // b = f % 2), of a stage of columns (K step f / kBF, block f % kBF / 2, b);
  // wavefront w requests fragments w, w + 8.
  const int frow = 8 * (l16 >> 2) + (l16 & 3);  // row of MFMA b: frow + 4 b
  const int voff_d = (frow * D + g8) * 2, voff_f = (frow * a.F + g8) * 2;
  const int wblk = wave / kBF, wks = wave % kBF / 2, wb = wave % 2;
  const int woff_d = (wblk * 32 * D + wb * 4 * D + wks * 32) * 2;
  const int woff_f = (wblk * 32 + (wks * 32 + wb * 4) * a.F) * 2;
  int cur = 1;  // the slot of the stage in use
  auto begin_stage = [&]() __attribute__((always_inline)) -> const bf16_t* {
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
    ring_barrier();
    cur ^= 1;
    return ring + cur * N::kStage;
  };
  // `blocks` 32-row blocks from row0 of a [*, D] weight
  auto request_rows = [&](const bf16_t* weight, int row0, int blocks) __attribute__((always_inline)) {
    const i32x4 rsrc = buffer_rsrc(weight);
    bf16_t* dst = ring + (cur ^ 1) * N::kStage + wave * kFrag;
#pragma unroll
    for (int i = 0; i < (kSB * kBF + kWaves - 1) / kWaves; ++i)
      if (wave + kWaves * i < blocks * kBF)
        enc_buffer_load_lds(rsrc, lds_ptr(dst + kWaves * i * kFrag), 16, voff_d,
                            row0 * D * 2 + woff_d + i * (kWaves / kBF) * 32 * D * 2, 0, 0);
  };
  // `blocks` 32-column blocks from col0 of a [D, F] weight
  auto request_cols = [&](const bf16_t* weight, int col0, int blocks) __attribute__((always_inline)) {
    const i32x4 rsrc = buffer_rsrc(weight);
    bf16_t* dst = ring + (cur ^ 1) * N::kStage + wave * kFrag;
#pragma unroll
    for (int i = 0; i < (kSB * kBF + kWaves - 1) / kWaves; ++i)
      if (wave + kWaves * i < blocks * kBF)
        enc_buffer_load_lds(rsrc, lds_ptr(dst + kWaves * i * kFrag), 16, voff_f,
                            col0 * 2 + woff_f + i * (kWaves / kBF) * 32 * 2, 0, 0);
  };
  request_rows(a.w[0][2], 0, kSB);
  // the first layer's vectors (and the table) are read before its first stage
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
  ring_barrier();
  const int hidden_blocks = min(kSB, a.F / 32);  // per FFN stage

#pragma unroll 1
  for (int layer = 0; layer < a.layers; ++layer) {
    const bf16_t* const* w = a.w[layer];
    const bf16_t* vec = vecs + (layer & 1) * N::kVecs;
    u32x4 h[kNB];
    row_norm<D>(x, vec + V::kG1, vec + V::kB1, a.eps, g8, h);
    u32x4 ctx[kNB];
#pragma unroll
    for (int c = 0; c < kNB; ++c) ctx[c] = u32x4{0u, 0u, 0u, 0u};

#pragma unroll 1
    for (int grp = 0; grp < N::kGroups; ++grp) {
        // ---- the group's Q stays in registers, its K and V^T go to LDS ----
      f32x4 a0, a1;
      u32x4 q[kNG];
#pragma unroll
      for (int i = 0; i < kQS; ++i) {
        const bf16_t* stage = begin_stage();
        // the next layer's vectors, into the block that everyone left before
        // this layer's first barrier
        if (i == 0 && grp == 0 && layer + 1 < a.layers)
          for (int v = wave; v < 8; v += kWaves)
            vec_to_lds<D>(vecs + ((layer + 1) & 1) * N::kVecs, a.w[layer + 1], v, a.F, lane);
        if (i + 1 < kQS)
          request_rows(w[2], grp * kGC + (i + 1) * 32 * kSB, kSB);
        else
          request_rows(w[2], D + grp * kGC, kSB);
#pragma unroll
        for (int j = 0; j < kSB; ++j) {
          block_product<D>(stage + j * kBF * kFrag, lane, h, a0, a1);
          q[i * kSB + j] = bias_pack(a0, a1, load16(vec + V::kQkv + grp * kGC + (i * kSB + j) * 32 + g8));
        }
      }
      const int kblk = keys.base + keys.q32;
#pragma unroll
      for (int i = 0; i < kQS; ++i) {
        const bf16_t* stage = begin_stage();
        if (i + 1 < kQS)
          request_rows(w[2], D + grp * kGC + (i + 1) * 32 * kSB, kSB);
        else
          request_rows(w[2], 2 * D + grp * kGC, kSB);
        // token t of the 32-token block is row 4 (t / 8) + t % 4 of fragment
        // (t / 4) % 2
        const int t = keys.qoff;
        bf16_t* kf = sK + ((2 * kblk + ((t >> 2) & 1)) * kNG + i * kSB) * kFrag + (4 * (t >> 3) + (t & 3) + 16 * g) * 8;
#pragma unroll
        for (int j = 0; j < kSB; ++j) {
          block_product<D>(stage + j * kBF * kFrag, lane, h, a0, a1);
          const u32x4 y = bias_pack(a0, a1, load16(vec + V::kQkv + D + grp * kGC + (i * kSB + j) * 32 + g8));
          if (live) *reinterpret_cast<u32x4*>(kf + j * kFrag) = y;
        }
      }
#pragma unroll
      for (int i = 0; i < kQS; ++i) {
        const bf16_t* stage = begin_stage();
        if (i + 1 < kQS)
          request_rows(w[2], 2 * D + grp * kGC + (i + 1) * 32 * kSB, kSB);
        else if (grp + 1 < N::kGroups)
          request_rows(w[2], (grp + 1) * kGC, kSB);
        else
          request_rows(w[4], 0, kSB);
        const int key = 16 * (qb & 1) + 4 * g;  // of the lane's first token, in its 32-key block
#pragma unroll
        for (int j = 0; j < kSB; ++j) {
          // V: the tokens are the A operand, so a lane holds the tokens 4 g ..
          // 4 g + 3 of channel frow + 4 b -- row l16 of V^T's fragment b
          const bf16_t* frags = stage + j * kBF * kFrag;
          const bf16_t* bias = vec + V::kQkv + 2 * D + grp * kGC + (i * kSB + j) * 32 + frow;
          f32x4 acc[2] = {zero4(), zero4()};
#pragma unroll
          for (int ks = 0; ks < kNB; ++ks) {
#pragma unroll
            for (int b = 0; b < 2; ++b)
              acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(h[ks]), lds_frag(frags, 2 * ks + b, lane), acc[b],
                                                               0, 0, 0);
          }
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            const float bb = bf16_to_f32(bias[4 * b]);
            if (live)
              *reinterpret_cast<u32x2*>(sV + (kblk * (kGC / 16) + 2 * (i * kSB + j) + b) * kFrag +
                                        (l16 + 16 * (key >> 3)) * 8 + (key & 7)) =
                  u32x2{pack_bf16x2(acc[b][0] + bb, acc[b][1] + bb), pack_bf16x2(acc[b][2] + bb, acc[b][3] + bb)};
          }
        }
      }
      // K and V^T of every wavefront (the ring's loads stay in flight)
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
      ring_barrier();

      // ---- attention: one head (four of 8 channels) per trip; the queries
      // are shifted down and the contexts in from the top, so that the loop
      // indexes registers statically ----
      constexpr int kChunk = HD < 32 ? 1 : HD / 32;  // chunks a trip takes
#pragma unroll 1
      for (int t = 0; t < kNG / kChunk; ++t) {
        u32x4 got[kChunk];
#pragma unroll
        for (int c = 0; c < kChunk; ++c) got[c] = u32x4{0u, 0u, 0u, 0u};
        if (attends) {
          if constexpr (HD >= 32) {
            bf16x8 qf[kChunk];
#pragma unroll
            for (int ks = 0; ks < kChunk; ++ks) qf[ks] = as_frag(q[ks]);
            head_attention<kGC, HD>(qf, sK, sV, t, keys, a.scale, lane, got);
          } else {
#pragma unroll 1
            for (int hh = 0; hh < 4; ++hh) {  // lane group hh holds head 4 t + hh's queries
              u32x4 mine, c8[1];
#pragma unroll
              for (int e = 0; e < 4; ++e) mine[e] = g == hh ? q[0][e] : 0u;
              const bf16x8 qf[1] = {as_frag(mine)};
              head_attention<kGC, HD>(qf, sK, sV, 4 * t + hh, keys, a.scale, lane, c8);
#pragma unroll
              for (int e = 0; e < 4; ++e) got[0][e] = g == hh ? c8[0][e] : got[0][e];
            }
          }
        }
#pragma unroll
        for (int c = 0; c + kChunk < kNG; ++c) q[c] = q[c + kChunk];
#pragma unroll
        for (int c = 0; c + kChunk < kNB; ++c) ctx[c] = ctx[c + kChunk];
#pragma unroll
        for (int c = 0; c < kChunk; ++c) ctx[kNB - kChunk + c] = got[c];
      }
      // (the next writes to K and V^T follow a stage's barrier, which every
      // wavefront reaches after its attention)
    }

    // ---- out_proj + residual (rows masked out keep x) ----
#pragma unroll
    for (int i = 0; i < kNB / kSB; ++i) {
      const bf16_t* stage = begin_stage();
      if (i + 1 < kNB / kSB)
        request_rows(w[4], (i + 1) * 32 * kSB, kSB);
      else
        request_rows(w[8], 0, hidden_blocks);
#pragma unroll
      for (int j = 0; j < kSB; ++j) {
        const int nb = i * kSB + j;
        f32x4 a0, a1;
        block_product<D>(stage + j * kBF * kFrag, lane, ctx, a0, a1);
        const u32x4 y = bias_residual(a0, a1, load16(vec + V::kOut + 32 * nb + g8), x[nb]);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[nb][e] = keep ? y[e] : x[nb][e];
      }
    }

    // ---- norm2, then the FFN + residual (rows masked out become 0): its
    // second product's K runs over the hidden features in order, so each 32
    // hidden features are consumed as they are produced ----
    row_norm<D>(x, vec + V::kG2, vec + V::kB2, a.eps, g8, h);
    f32x4 o[kNB][2];
#pragma unroll
    for (int ob = 0; ob < kNB; ++ob) {
      o[ob][0] = zero4();
      o[ob][1] = zero4();
    }
#pragma unroll 1
    for (int f0 = 0; f0 < a.F; f0 += 32 * kSB) {
      const bf16_t* stage = begin_stage();
      request_cols(w[10], f0, hidden_blocks);
      bf16x8 hf[kSB];
#pragma unroll
      for (int j = 0; j < kSB; ++j) {
        if (j >= hidden_blocks) continue;
        f32x4 a0, a1;
        block_product<D>(stage + j * kBF * kFrag, lane, h, a0, a1);
        hf[j] = as_frag(gelu8(bias_pack(a0, a1, load16(vec + V::kFfnIn + f0 + 32 * j + g8)),
                              reinterpret_cast<const char*>(gelu), table));
      }
      stage = begin_stage();
      if (f0 + 32 * kSB < a.F)
        request_rows(w[8], f0 + 32 * kSB, hidden_blocks);
      else if (layer + 1 < a.layers)
        request_rows(a.w[layer + 1][2], 0, kSB);
#pragma unroll
      for (int j = 0; j < kSB; ++j) {
        if (j >= hidden_blocks) continue;
#pragma unroll
        for (int ob = 0; ob < kNB; ++ob) {
#pragma unroll
          for (int b = 0; b < 2; ++b)
            o[ob][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lds_frag(stage, j * kBF + 2 * ob + b, lane), hf[j],
                                                               o[ob][b], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int c = 0; c < kNB; ++c) {
      const u32x4 y = bias_residual(o[c][0], o[c][1], load16(vec + V::kFfnOut + 32 * c + g8), x[c]);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[c][e] = keep ? y[e] : 0u;
    }
  }

  if (a.final_g != nullptr) {
    u32x4 y[kNB];
    row_norm<D>(x, a.final_g, a.final_b, a.eps, g8, y);
#pragma unroll
    for (int c = 0; c < kNB; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) x[c][e] = keep ? y[c][e] : 0u;
  }
  if (live) {
#pragma unroll
    for (int c = 0; c < kNB; ++c) *reinterpret_cast<u32x4*>(a.out + row * D + 32 * c + g8) = x[c];
  }
}

// Sequences of a workgroup: as many as its wavefronts (16 tokens each) and its
// four 32-key blocks hold.
int64_t sequences_per_group(int64_t S) {
  const int64_t by_waves = kWaves / ((S + 15) / 16), by_keys = 4 / ((S + 31) / 32);
  return by_waves < by_keys ? by_waves : by_keys;
}

template <int D, int HD>
hipError_t launch(const NarrowArgs& a, hipStream_t st) {
  auto kernel = narrow_forward_kernel<D, HD>;
  constexpr int kLds = Narrow<D, HD>::kLds;
  if constexpr (kLds > 64 * 1024) {
    // above 64 KiB of dynamic LDS the kernel has to opt in (once per process)
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (attr != hipSuccess) return attr;
  }
  const int64_t per_group = sequences_per_group(a.S);
  const int64_t groups = (a.B + per_group - 1) / per_group;
  hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(groups)), dim3(kWaves * kWave), kLds, st, a);
  return hipGetLastError();
}

}  // namespace

bool narrow_forward_supported(int64_t S, int64_t D, int64_t H, int64_t F) {
  auto narrow = [](int64_t v) { return v == 32 || v == 64 || v == 128; };
  const int64_t hd = D / H;
  return S >= 1 && S <= 128 && narrow(D) && narrow(F) && D % H == 0 && (hd == 8 || narrow(hd));
}

// Where one launch beats three launches a layer (narrow_rows.hip), measured on
// MI355X over 1 to 128 tokens a sequence and 1 to 20000 sequences, two layers, ffn
// 128, us (three a layer / one; batch x tokens).  The launches' time hardly moves
// up to a few thousand tokens and then grows with the attention's workgroups, one
// per sequence and head even where a sequence is a token, ragged tiles costing more
// than whole ones; one launch's hardly moves up to 256 workgroups of at most four
// sequences, and grows with the heads, which a wavefront takes one after the other,
// with the 32-key blocks and with ffn_dim (2 a layer less at 64, 3 at 32):
//   d_model 32 and 64, 32 channels a head and more: always (d 64, hd 32: 8 x 128
//     27.6 / 28.4, 128 x 64 37.5 / 25.3, 65536 x 1 2248 / 762);
//   hd 8 at d 32: 32 x 128 29.2 / 34.8, 128 x 64 34.8 / 27.7; at d 64: 96 x 16
//     34.0 / 35.1, 160 x 16 43.6 / 35.1, 160 x 65 60.9 / 55.9; at d 128: 128 x 64
//     75.6 / 114, 192 x 24 89.5 / 91.7, 512 x 16 173 / 80.6, 65536 x 1 16561 / 3363;
//   d 128, hd 32: 192 x 4 38.9 / 44.4, 240 x 12 47.1 / 45.2, 160 x 24 43.3 / 48.9,
//     192 x 32 54.0 / 49.7, 96 x 64 48.5 / 54.8, 160 x 64 64.6 / 54.7, 64 x 128 53.2
//     / 62.1, 96 x 128 71.6 / 62.3;
//   d 128, hd 64: 128 x 12 36.9 / 38.6, 64 x 40 40.3 / 42.7, 128 x 40 52.4 / 42.8,
//     64 x 64 38.1 / 44.7, 96 x 64 49.8 / 44.7; ffn 32 102 x 33 43.7 / 36.8;
//   d 128, hd 128, one workgroup per CU: 320 x 2 40.8 / 44.2, 96 x 40 48.0 / 47.8,
//     128 x 40 57.0 / 48.3, 64 x 64 37.3 / 49.0, 128 x 64 48.4 / 49.5; in many
//     rounds of workgroups that are mostly padding, or whose wavefronts all have
//     128 keys, 1321 x 1 71 / 78, 2048 x 1 98 / 88, 16384 x 1 567 / 678, 512 x 128
//     120 / 107, 1024 x 128 194 / 214; ffn 64 2629 x 4 142 / 117.
bool narrow_forward_faster(int64_t B, int64_t S, int64_t D, int64_t H, int64_t F) {
  const int64_t hd = D / H;
  if (hd == 8) return D == 32 ? B >= 48 || S <= 64 : B >= (D == 128 ? 240 : S <= 16 ? 112 : 160);
  if (D < 128) return true;
  if (hd == 32) return B >= (S <= 16 ? 100 + F : S <= 32 ? 150 + F / 3 : S <= 64 ? 120 + F / 5 : 70 + F / 7);
  const bool whole = S % 64 == 0;
  if (hd == 64) return S <= 16 ? B >= 64 + 3 * F / 4 : B * S >= (whole ? 3800 + 12 * F : S <= 64 ? 34 * F : 4100);
  const int64_t groups = (B + sequences_per_group(S) - 1) / sequences_per_group(S);
  // (up to eight tokens: 36 us and 1/16 of ffn_dim a round of 256 workgroups,
  // against 36 and 0.033 to 0.04 a sequence)
  if (S <= 8)
    return B >= (S <= 2 ? 224 : 112) + F && (36 + F / 16) * ((groups + 255) / 256) <= 36 + B * (32 + S) / 1000;
  if (S <= 16) return B >= F;
  return B * S >= (whole ? 5000 + 13 * F : S <= 64 ? 32 * F : 4100) && (S <= 64 || groups <= 768);
}

hipError_t narrow_forward_bf16(const NarrowForward& f, hipStream_t st) {
  if (!narrow_forward_supported(f.S, f.D, f.H, f.F) || f.layers < 1 || f.B >= (int64_t(1) << 31)) return hipErrorInvalidValue;
  NarrowArgs a;
  hipError_t e = gemm_gelu_table(st, &a.gelu_table, &a.gelu_ready);
  if (e != hipSuccess) return e;
  a.kv_len = f.kv_len;
  a.key_mask = f.key_mask;
  a.row_mask = f.row_mask;
  a.B = static_cast<int>(f.B);
  a.S = static_cast<int>(f.S);
  a.F = static_cast<int>(f.F);
  a.causal = f.causal ? 1 : 0;
  a.eps = f.eps;
  a.scale = f.scale;
  // more layers than a launch's argument block holds: several launches, the
  // later ones in place (a wavefront reads and writes only its own tokens)
  for (int64_t first = 0; first < f.layers; first += kNarrowMaxLayers) {
    const int64_t count = f.layers - first < kNarrowMaxLayers ? f.layers - first : kNarrowMaxLayers;
    const bool last = first + count == f.layers;
    a.x = first == 0 ? f.x : f.out;
    a.out = f.out;
    a.layers = static_cast<int>(count);
    a.final_g = last ? f.final_g : nullptr;
    a.final_b = last ? f.final_b : nullptr;
    for (int64_t l = 0; l < count; ++l)
      for (int i = 0; i < 12; ++i) a.w[l][i] = static_cast<const bf16_t*>(f.weights[(first + l) * 12 + i]);
    switch (f.D * 1000 + f.D / f.H) {
      case 32008: e = launch<32, 8>(a, st); break;
      case 32032: e = launch<32, 32>(a, st); break;
      case 64008: e = launch<64, 8>(a, st); break;
      case 64032: e = launch<64, 32>(a, st); break;
      case 64064: e = launch<64, 64>(a, st); break;
      case 128008: e = launch<128, 8>(a, st); break;
      case 128032: e = launch<128, 32>(a, st); break;
      case 128064: e = launch<128, 64>(a, st); break;
      case 128128: e = launch<128, 128>(a, st); break;
      default: return hipErrorInvalidValue;
    }
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace enc
