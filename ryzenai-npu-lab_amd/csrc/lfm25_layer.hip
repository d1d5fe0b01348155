// One token through one decoder layer as the reference's per-operation
// programs split it (recurrent block; attention prefix, context + cache,
// tail), a launch per dependent product. These calls get their weights from
// HBM and run alone, so what bounds them is launches (2.5 us each back to
// back, more from Python) and each product's first load; every element-wise
// step rides in the product that feeds it:
//
//   conv_in   operator norm + in_proj + gated short conv (+ state, taps)
//   prefix    operator norm + q | k | v + QK norm + RoPE (+ hidden copy)
//   scores    s_j, their block statistics, the grown cache, the hidden copy
//   context   softmax and sum of values
//   project   W x + residual (out_proj, o_proj and w2)
//   up        ffn norm + w1, w3 + SiLU gate
//
// Each product's rows are spread so that every CU gets the same bytes, a
// wave requests its weight rows before the activation they meet, and row sums
// add in the order of the plain GEMV (lfm25_ops.hip), so those bits are its.
#include "lfm25_host.h"
#include "lfm25_stages.h"

namespace lfm25 {
namespace {

// R weight rows of K values, in flight.
template <int K, int R>
struct Rows {
  static constexpr int kChunks = LaneVec<K>::kChunks;
  Pack8 w[R][kChunks];
  __device__ __forceinline__ void load(int r, const uint16_t* row) {
#pragma unroll
    for (int c = 0; c < kChunks; ++c) w[r][c] = load8_stream(row + c * 512 + lane_id() * 8);
  }
  __device__ __forceinline__ float dot(int r, const LaneVec<K>& x) const {
    float acc = 0.0f;
#pragma unroll
    for (int c = 0; c < kChunks; ++c) acc = fma8(w[r][c], x.v + c * 8, acc);
    return wave_sum(acc);
  }
};

constexpr int kWaves = 4;  // per block of the 256-block products

// out[r] = bf16(residual[r] + bf16(W[r] . x)), a wave per row of 1,024.
template <int K>
__global__ void __launch_bounds__(kWaves* kWave) k_layer_project(const uint16_t* __restrict__ w,
                                                                 const uint16_t* __restrict__ x,
                                                                 const uint16_t* __restrict__ residual,
                                                                 uint16_t* __restrict__ out) {
  const int r = blockIdx.x * kWaves + wave_id();
  Rows<K, 1> rows;
  rows.load(0, w + (size_t)r * K);
  LaneVec<K> v;
  load_lane_vec<K>(x, v);
  const float res = bf16_to_f32(residual[r]);
  const float d = rows.dot(0, v);
  if (lane_id() == 0) out[r] = f32_to_bf16(res + round_bf16(d));
}

// g[f] = bf16(bf16(silu(bf16(w1[f] . n))) * bf16(w3[f] . n)), n = RMSNorm(h):
// 256 blocks of five waves, two columns a wave, so that the 2,560 columns are
// ten to a CU.
constexpr int kUpWaves = 5, kUpCols_ = 2;
static_assert(256 * kUpWaves * kUpCols_ == kFfn, "ten columns per block");
__global__ void __launch_bounds__(kUpWaves* kWave) k_layer_up(const uint16_t* __restrict__ h,
                                                              const uint16_t* __restrict__ gamma,
                                                              const uint16_t* __restrict__ w1,
                                                              const uint16_t* __restrict__ w3,
                                                              uint16_t* __restrict__ g) {
  const int f = (blockIdx.x * kUpWaves + wave_id()) * kUpCols_;
  Rows<kHidden, 2 * kUpCols_> rows;
#pragma unroll
  for (int j = 0; j < kUpCols_; ++j) {
    rows.load(2 * j, w1 + (size_t)(f + j) * kHidden);
    rows.load(2 * j + 1, w3 + (size_t)(f + j) * kHidden);
  }
  LaneVec<kHidden> v;
  load_lane_vec<kHidden>(h, v);
  rms_norm_lane_vec<kHidden>(v, gamma);
#pragma unroll
  for (int j = 0; j < kUpCols_; ++j) {
    const float a = rows.dot(2 * j, v), b = rows.dot(2 * j + 1, v);
    if (lane_id() == j) g[f + j] = f32_to_bf16(silu_bf16(round_bf16(a)) * round_bf16(b));
  }
}

// y = the gated short conv of RMSNorm(hidden): a wave per channel (rows c,
// 1024 + c, 2048 + c of in_proj are its B, C and x). state and taps are
// [1024 x 3] each; next = [next state | taps].
__global__ void __launch_bounds__(kWaves* kWave) k_layer_conv_in(const uint16_t* __restrict__ hidden,
                                                                 const uint16_t* __restrict__ gamma,
                                                                 const uint16_t* __restrict__ w_in,
                                                                 const uint16_t* state, const uint16_t* taps,
                                                                 uint16_t* next, uint16_t* __restrict__ y) {
  const int c = blockIdx.x * kWaves + wave_id();
  Rows<kHidden, 3> rows;
#pragma unroll
  for (int j = 0; j < 3; ++j) rows.load(j, w_in + (size_t)(j * kHidden + c) * kHidden);
  uint16_t st[kConvTaps], tap[kConvTaps];
#pragma unroll
  for (int j = 0; j < kConvTaps; ++j) {
    st[j] = state[c * kConvTaps + j];
    tap[j] = taps[c * kConvTaps + j];
  }
  LaneVec<kHidden> v;
  load_lane_vec<kHidden>(hidden, v);
  rms_norm_lane_vec<kHidden>(v, gamma);
  const float b = rows.dot(0, v), g = rows.dot(1, v), x = rows.dot(2, v);
  if (lane_id() == 0) {
    y[c] = f32_to_bf16(conv_gate_channel(round_bf16(b), round_bf16(g), round_bf16(x), tap, st, st));
#pragma unroll
    for (int j = 0; j < kConvTaps; ++j) {
      next[c * kConvTaps + j] = st[j];
      next[(kHidden + c) * kConvTaps + j] = tap[j];
    }
  }
}

// One head of q | k | v per block (16 q, 8 k, 8 v; 16 waves of four rows), the
// q and k heads through QK norm and RoPE (aux = [q_gamma | k_gamma | cos |
// sin]); with_hidden: out[2048 ..] = hidden, an eighth per v block.
constexpr int kPrefixThreads = 1024;
__global__ void __launch_bounds__(kPrefixThreads) k_layer_prefix(const uint16_t* __restrict__ hidden,
                                                                 const uint16_t* __restrict__ gamma,
                                                                 const uint16_t* __restrict__ w,
                                                                 const uint16_t* __restrict__ aux,
                                                                 uint16_t* __restrict__ out, int with_hidden) {
  constexpr int R = kHeadDim * kWave / kPrefixThreads;  // rows per wave
  __shared__ float raw[kHeadDim];
  const int head = blockIdx.x, wv = wave_id(), l = lane_id();
  Rows<kHidden, R> rows;
#pragma unroll
  for (int r = 0; r < R; ++r) rows.load(r, w + (size_t)(head * kHeadDim + R * wv + r) * kHidden);
  LaneVec<kHidden> v;
  load_lane_vec<kHidden>(hidden, v);
  rms_norm_lane_vec<kHidden>(v, gamma);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float d = rows.dot(r, v);
    if (l == 0) raw[R * wv + r] = round_bf16(d);
  }
  __syncthreads();
  if (wv == 0) {
    float o = raw[l];
    if (head < kHeads + kKvHeads)
      o = norm_rope_lane(o, bf16_to_f32(aux[(head < kHeads ? 0 : kHeadDim) + l]), bf16_to_f32(aux[2 * kHeadDim + l]),
                         bf16_to_f32(aux[3 * kHeadDim + l]));
    out[head * kHeadDim + l] = f32_to_bf16(o);
  } else if (wv < 3 && with_hidden && head >= kHeads + kKvHeads) {
    const int e = (head - kHeads - kKvHeads) * (kHidden / kKvHeads) + (wv - 1) * kWave + l;
    out[2 * kHidden + e] = hidden[e];
  }
}

// ------------------------------------------------------------------ attention
//
// Decode attention over `past` cached positions and the current one, eager
// semantics (attn_core_t, lfm25_stages.h), with the cache grown by a row:
// caches hold, per KV head, keys [P x 64] then values. One block per head
// walked its 256 KB at 1,023 positions alone (8 of 256 CUs). Here the scores
// run a block per head and 64 positions, which also copies those rows into
// the next cache; the probabilities need the statistics of all of them, so
// the values follow in a second launch, a block per head and 16 dimensions.

constexpr int kScorePos = 64;
constexpr int kValueThreads = 1024;
constexpr int kValueDims = 16;  // dimensions per block
struct AttWorkspace {
  float2 stats[kKvHeads][2][kMaxCapacity / kScorePos];  // (maximum, sum of e^(s - maximum)) per block
  float scores[kKvHeads][2][kMaxCapacity];
};

__global__ void __launch_bounds__(256) k_layer_scores(const uint16_t* __restrict__ qkv,
                                                      const uint16_t* __restrict__ cache,
                                                      uint16_t* __restrict__ tail, uint16_t* __restrict__ next,
                                                      AttWorkspace* __restrict__ ws, int past) {
  __shared__ float2 part[2][4];
  const int h = blockIdx.x, chunk = blockIdx.y, t = threadIdx.x;
  // four threads per position, 16 dimensions each
  const int j = chunk * kScorePos + t / 4, d0 = 16 * (t % 4);
  const bool in = j <= past;
  uint4 k[2], v[2];
  {
    const uint16_t* row = cache + (size_t)h * 2 * past * kHeadDim + (size_t)min(j, past - 1) * kHeadDim + d0;
    const uint16_t* kr = j < past ? row : qkv + kHidden + h * kHeadDim + d0;
    const uint16_t* vr = j < past ? row + (size_t)past * kHeadDim : qkv + kHidden + kKvHeads * kHeadDim + h * kHeadDim + d0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      k[i] = reinterpret_cast<const uint4*>(kr)[i];
      v[i] = reinterpret_cast<const uint4*>(vr)[i];
    }
  }
  uint4 q[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int i = 0; i < 2; ++i) q[a][i] = reinterpret_cast<const uint4*>(qkv + (2 * h + a) * kHeadDim + d0)[i];
  if (in) {
    uint4* dst = reinterpret_cast<uint4*>(next + ((size_t)h * 2 * (past + 1) + j) * kHeadDim + d0);
    uint4* dv = reinterpret_cast<uint4*>(next + ((size_t)(h * 2 + 1) * (past + 1) + j) * kHeadDim + d0);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      dst[i] = k[i];
      dv[i] = v[i];
    }
  }
  if (chunk == 0 && t < kHidden / kKvHeads) {
    const int e = h * (kHidden / kKvHeads) + t;
    tail[e] = qkv[2 * kHidden + e];
  }
  float kf[16];
  unpack8(Pack8{{k[0].x, k[0].y, k[0].z, k[0].w}}, kf);
  unpack8(Pack8{{k[1].x, k[1].y, k[1].z, k[1].w}}, kf + 8);
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    float qf[16];
    unpack8(Pack8{{q[a][0].x, q[a][0].y, q[a][0].z, q[a][0].w}}, qf);
    unpack8(Pack8{{q[a][1].x, q[a][1].y, q[a][1].z, q[a][1].w}}, qf + 8);
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) s = fmaf(qf[i], kf[i], s);
    s += dpp_f32<kDppQuadXor1>(s);
    s += dpp_f32<kDppQuadXor2>(s);
    s = round_bf16(s) * 0.125f;
    if (in && t % 4 == 0) ws->scores[h][a][j] = s;
    // each position's score sits in four lanes: the sum counts it once
    const float m = wave_max(in ? s : -INFINITY);
    const float z = wave_sum(in && t % 4 == 0 ? expf(s - m) : 0.0f);
    if (lane_id() == 0) part[a][wave_id()] = float2{m, z};
  }
  __syncthreads();
  if (t < 2) {
    float m = part[t][0].x;
#pragma unroll
    for (int w = 1; w < 4; ++w) m = fmaxf(m, part[t][w].x);
    float z = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w)
      if (part[t][w].x != -INFINITY) z += part[t][w].y * expf(part[t][w].x - m);  // (a wave past the last position)
    ws->stats[h][t][chunk] = float2{m, z};
  }
}

__global__ void __launch_bounds__(kValueThreads) k_layer_context(const uint16_t* __restrict__ next,
                                                                 const AttWorkspace* __restrict__ ws,
                                                                 uint16_t* __restrict__ context, int past) {
  __shared__ float sum[kValueThreads / kWave][2][kValueDims];
  const int h = blockIdx.x, d0 = blockIdx.y * kValueDims, l = lane_id();
  const int total = past + 1, chunks = (total + kScorePos - 1) / kScorePos;
  // a wave takes 32 positions, half its lanes the first 8 of the block's
  // dimensions and half the other 8; the block 512 positions a pass
  constexpr int kPer = kValueThreads / 2;
  const int slot = 32 * wave_id() + (l & 31), e0 = d0 + 8 * (l >> 5);
  const uint16_t* values = next + (size_t)(h * 2 + 1) * total * kHeadDim + e0;
  const float *s0 = ws->scores[h][0], *s1 = ws->scores[h][1];
  // the first two passes' rows and scores are requested before the statistics
  // are waited for: at up to 1,024 positions one round of loads is all
  Pack8 vr[2];
  float sr[2][2];
  const auto load = [&](int base) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int jc = min(base + u * kPer + slot, past);
      vr[u] = load8(values + (size_t)jc * kHeadDim);
      sr[u][0] = s0[jc];
      sr[u][1] = s1[jc];
    }
  };
  load(0);
  float m[2], z[2];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    // (at most 64 blocks of positions: a lane each)
    const float2 s = l < chunks ? ws->stats[h][a][l] : float2{-INFINITY, 0.0f};
    m[a] = wave_max(s.x);
    z[a] = wave_sum(l < chunks ? s.y * expf(s.x - m[a]) : 0.0f);
  }
  float c[2][8];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int i = 0; i < 8; ++i) c[a][i] = 0.0f;
  for (int base = 0; base < total; base += 2 * kPer) {
    if (base > 0) load(base);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const bool in = base + u * kPer + slot < total;
      float vf[8];
      unpack8(vr[u], vf);
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const float p = round_bf16(expf(sr[u][a] - m[a]) / z[a]);
#pragma unroll
        for (int e = 0; e < 8; ++e) c[a][e] = in ? fmaf(p, vf[e], c[a][e]) : c[a][e];
      }
    }
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float r = row16_sum(c[a][e]);
      const float half = l < 32 ? lane_value(r, 0) + lane_value(r, 16) : lane_value(r, 32) + lane_value(r, 48);
      if ((l & 31) == 0) sum[wave_id()][a][8 * (l >> 5) + e] = half;
    }
  __syncthreads();
  const int t = threadIdx.x;
  if (t < 2 * kValueDims) {
    const int a = t / kValueDims, d = t % kValueDims;
    float s = sum[0][a][d];
#pragma unroll
    for (int w = 1; w < kValueThreads / kWave; ++w) s += sum[w][a][d];
    context[(2 * h + a) * kHeadDim + d0 + d] = f32_to_bf16(s);
  }
}

// h = residual + W x; out = h + w2 . gate(norm(h)): the second half of a layer.
struct Mlp {
  const uint16_t *gamma, *w1, *w3, *w2;
};
int layer_tail(const uint16_t* w, const uint16_t* x, const uint16_t* residual, const Mlp& m, uint16_t* out,
               uint16_t* ws, hipStream_t s, const char* what) {
  uint16_t *h = ws, *g = ws + kHidden;
  k_layer_project<kHidden><<<kHidden / kWaves, kWaves * kWave, 0, s>>>(w, x, residual, h);
  k_layer_up<<<256, kUpWaves * kWave, 0, s>>>(h, m.gamma, m.w1, m.w3, g);
  k_layer_project<kFfn><<<kHidden / kWaves, kWaves * kWave, 0, s>>>(m.w2, g, h, out);
  return check_launch(what);
}
constexpr int kGammaTile = 4096;
constexpr size_t kTailBytes = (size_t)(kHidden + kFfn) * 2;
Mlp mlp_at(const uint16_t* p) {  // [ffn gamma tile | w1 | w3 | w2]
  const uint16_t* w = p + kGammaTile;
  return Mlp{p, w, w + (size_t)kFfn * kHidden, w + (size_t)2 * kFfn * kHidden};
}

}  // namespace
}  // namespace lfm25

using namespace lfm25;

extern "C" {

size_t lfm25_layer_workspace_bytes(void) {
  return sizeof(AttWorkspace) > kTailBytes + kHidden * 2 ? sizeof(AttWorkspace) : kTailBytes + kHidden * 2;
}

int lfm25_recurrent_block(const uint16_t* hidden, const uint16_t* state, const uint16_t* conv_weight,
                          const uint16_t* packed_weights, uint16_t* next_state_and_weight, uint16_t* block_output,
                          void* workspace, lfm25_stream_t stream) {
  LFM25_REQUIRE(hidden && state && conv_weight && packed_weights && next_state_and_weight && block_output && workspace,
                "recurrent_block: null pointer");
  LFM25_REQUIRE(aligned16(hidden) && aligned16(packed_weights) && aligned16(workspace),
                "recurrent_block: hidden, weights and workspace must be 16-byte aligned");
  uint16_t* y = static_cast<uint16_t*>(workspace);
  const uint16_t* w_in = packed_weights + kGammaTile;
  const uint16_t* w_out = w_in + (size_t)3 * kHidden * kHidden;
  k_layer_conv_in<<<kHidden / kWaves, kWaves * kWave, 0, stream>>>(hidden, packed_weights, w_in, state, conv_weight,
                                                                   next_state_and_weight, y);
  return layer_tail(w_out, y, hidden, mlp_at(w_out + (size_t)kHidden * kHidden), block_output, y + kHidden, stream,
                    "recurrent_block");
}

int lfm25_attention_prefix(const uint16_t* hidden, const uint16_t* packed_gamma_and_weight, const uint16_t* aux,
                           uint16_t* qkv_output, int32_t include_hidden, lfm25_stream_t stream) {
  LFM25_REQUIRE(hidden && packed_gamma_and_weight && aux && qkv_output, "attention_prefix: null pointer");
  LFM25_REQUIRE(aligned16(hidden) && aligned16(packed_gamma_and_weight), "attention_prefix: 16-byte alignment");
  k_layer_prefix<<<kHeads + 2 * kKvHeads, kPrefixThreads, 0, stream>>>(
      hidden, packed_gamma_and_weight, packed_gamma_and_weight + kGammaTile, aux, qkv_output, include_hidden);
  return check_launch("attention_prefix");
}

int lfm25_attention_context_cache(const uint16_t* qkv_and_hidden, const uint16_t* past_cache,
                                  uint16_t* packed_tail_input, uint16_t* next_cache, int32_t past_length,
                                  void* workspace, lfm25_stream_t stream) {
  LFM25_REQUIRE(qkv_and_hidden && past_cache && packed_tail_input && next_cache && workspace,
                "attention_context_cache: null pointer");
  LFM25_REQUIRE(past_length >= 1 && past_length < kMaxCapacity,
                "attention_context_cache: past_length must be in [1, %d), got %d", kMaxCapacity, past_length);
  LFM25_REQUIRE(aligned16(qkv_and_hidden) && aligned16(past_cache) && aligned16(next_cache) && aligned16(workspace),
                "attention_context_cache: qkv_and_hidden, the caches and the workspace must be 16-byte aligned");
  AttWorkspace* ws = static_cast<AttWorkspace*>(workspace);
  const int chunks = past_length / kScorePos + 1;
  k_layer_scores<<<dim3(kKvHeads, chunks), 256, 0, stream>>>(qkv_and_hidden, past_cache, packed_tail_input, next_cache,
                                                             ws, past_length);
  k_layer_context<<<dim3(kKvHeads, kHeadDim / kValueDims), kValueThreads, 0, stream>>>(
      next_cache, ws, packed_tail_input + kHidden, past_length);
  return check_launch("attention_context_cache");
}

int lfm25_attention_tail(const uint16_t* packed_hidden_and_context, const uint16_t* packed_weights,
                         uint16_t* block_output, void* workspace, lfm25_stream_t stream) {
  LFM25_REQUIRE(packed_hidden_and_context && packed_weights && block_output && workspace,
                "attention_tail: null pointer");
  LFM25_REQUIRE(aligned16(packed_hidden_and_context) && aligned16(packed_weights) && aligned16(workspace),
                "attention_tail: inputs and workspace must be 16-byte aligned");
  return layer_tail(packed_weights, packed_hidden_and_context + kHidden, packed_hidden_and_context,
                    mlp_at(packed_weights + (size_t)kHidden * kHidden), block_output, static_cast<uint16_t*>(workspace),
                    stream, "attention_tail");
}

}  // extern "C"
