// The prompt pass on gfx950: the rows of one or more prompts (up to 4,096
// rows, each prompt a run of consecutive positions of its sequence) through
// all 14 layers as matrix-matrix products, on the batched pass's KV caches
// and conv states (lfm25_batch.hip, whose passes stop at 64 rows because
// they keep every row in one block's LDS). It is the reference's batched
// prompt pass (prefill_design, experiments/lfm25_x8.py:341-416) with a prompt
// per pass instead of PB = 4 tokens.
//
// At 64 rows a pass the prompt's time was the weights: 1,024 tokens read the
// 325 MB of layers sixteen times, 15.6 ms, in 94 small kernels each time.
// Here each weight tile multiplies every row (lfm25_gemm.h) and a layer is
// seven or eight launches whatever the prompt's length:
//
//   conv layer: in_proj product -> conv gate -> out_proj product + residual
//   attention:  q|k|v product -> QK norm + RoPE + append -> attention ->
//               o_proj product + residual
//   both:       norm -> w1 | w3 product with the SiLU gate -> w2 product +
//               residual -> norm (of the next layer)
//
// Rounding points are the batched pass's (and the decode's): BF16 at every
// projection's output, norm, gate and residual, FP32 inside.
#include <algorithm>

#include "lfm25_ahead.h"
#include "lfm25_gemm.h"
#include "lfm25_host.h"
#include "lfm25_layout.h"
#include "lfm25_stages.h"

namespace lfm25 {
namespace {

typedef tile::bf16x8 bf16x8;
typedef tile::f32x4 f32x4;

// Workspace for `rows` rows, in bytes: x, xn, y [rows][1024], big [rows][3072]
// (in_proj, or q|k|v in 2,048, or the 2,560 gate values), the row table.
constexpr size_t kPpRowBytes = (size_t)(3 * kHidden + 3 * kHidden) * 2 + sizeof(int4);

// A row's sequence and position; chunk = its index within its run; to_end =
// the rows of its run that follow it.
struct Row {
  int seq, pos, chunk, to_end;
};

struct Prompt {
  const uint16_t* weights;
  const uint16_t* embedding;
  const uint16_t* rope;
  uint16_t* conv_state;   // [seqs][8][1024][3]
  uint16_t* key_cache;    // [seqs][6][8][capacity][64]
  uint16_t* value_cache;
  uint16_t *x, *xn, *y, *big;
  Row* table;
  int32_t* status;
  int rows, capacity, vocab;
};

__device__ __forceinline__ size_t pp_kv_base(const Prompt& p, int seq, int att, int g) {
  return ((size_t)(seq * LFM25_ATTN_LAYERS + att) * kKvHeads + g) * p.capacity * kHeadDim;
}

using tile::pack_pair;

// ------------------------------------------------------------------ norms

constexpr int kNormRows = 4;  // rows (waves) per block

// A wave's row (LaneVec) as BF16.
__device__ __forceinline__ void store_lane_vec(uint16_t* row, const LaneVec<kHidden>& v) {
#pragma unroll
  for (int c = 0; c < LaneVec<kHidden>::kChunks; ++c)
    *reinterpret_cast<uint4*>(row + c * 512 + lane_id() * 8) =
        uint4{pack_pair(v.v[8 * c], v.v[8 * c + 1]), pack_pair(v.v[8 * c + 2], v.v[8 * c + 3]),
              pack_pair(v.v[8 * c + 4], v.v[8 * c + 5]), pack_pair(v.v[8 * c + 6], v.v[8 * c + 7])};
}

// Row m of x = the embedding row of its token (ids outside the table are
// clamped and flagged in status bit 0), xn = its RMSNorm with the first
// layer's operator norm; and the row's entry of the row table.
__global__ void __launch_bounds__(kNormRows* kWave) k_pp_embed(Prompt p, PromptRuns runs,
                                                               const int32_t* __restrict__ tokens) {
  const int m = blockIdx.x * kNormRows + wave_id();
  if (m >= p.rows) return;
  int r = 0, first = 0;
  while (m >= first + runs.run[r].count) first += runs.run[r++].count;
  if (lane_id() == 0)
    p.table[m] = Row{runs.run[r].sequence, runs.run[r].position + m - first, m - first, first + runs.run[r].count - 1 - m};
  int tok = tokens[m];
  if (tok < 0 || tok >= p.vocab) {
    if (lane_id() == 0) atomicOr(p.status, 1);
    tok = tok < 0 ? 0 : p.vocab - 1;
  }
  LaneVec<kHidden> v;
  load_lane_vec<kHidden>(p.embedding + (size_t)tok * kHidden, v);
  store_lane_vec(p.x + (size_t)m * kHidden, v);
  rms_norm_lane_vec<kHidden>(v, conv_tensor<C_OPNORM>(p.weights, 0));
  store_lane_vec(p.xn + (size_t)m * kHidden, v);
}

// xn = RMSNorm of x, one wave per row (Lfm2RMSNorm.forward,
// modeling_lfm2.py:54-59, two roundings).
__global__ void __launch_bounds__(kNormRows* kWave) k_pp_norm(const uint16_t* __restrict__ x,
                                                              const uint16_t* __restrict__ gamma,
                                                              uint16_t* __restrict__ xn, int rows) {
  const int m = blockIdx.x * kNormRows + wave_id();
  if (m >= rows) return;
  LaneVec<kHidden> v;
  load_lane_vec<kHidden>(x + (size_t)m * kHidden, v);
  rms_norm_lane_vec<kHidden>(v, gamma);
  store_lane_vec(xn + (size_t)m * kHidden, v);
}

// ------------------------------------------------------------------ products

enum PpEpi { PP_STORE, PP_RESIDUAL, PP_SILU };

struct PpGemm {
  const uint16_t* a;  // [rows][k]
  const uint16_t* w;  // [n][k] (PP_SILU: w1 and w3, n / 2 rows each, back to back)
  uint16_t* c;        // [rows][ldc]
  int rows, n, k, ldc;
  tile::Tiles tiles;
  AheadPair ahead;  // weights of the products to come
};

// PP_STORE: c = bf16(a . w^T). PP_RESIDUAL: c = bf16(c + bf16(a . w^T)) (the
// residual add of Lfm2DecoderLayer.forward, modeling_lfm2.py:431). PP_SILU: c =
// bf16(bf16(silu(bf16(w1 . a))) * bf16(w3 . a)) (Lfm2MLP.forward,
// modeling_lfm2.py:135-136): a lane's run of kLaneN columns is half rows of w1
// and half the same rows of w3, so both of a gate's products end in one lane.
template <int EPI, typename S>
__global__ void __launch_bounds__(S::kThreads, 2) k_pp_gemm(const PpGemm g) {
  extern __shared__ __attribute__((aligned(16))) char lds_raw[];
  auto& sh = *reinterpret_cast<tile::Lds<S>*>(lds_raw);
  const int own = g.tiles.blocks();
  if ((int)blockIdx.x >= own) return read_ahead(g.ahead, own);
  int tm, tn;
  if (!g.tiles.of(blockIdx.x, tm, tn)) return;
  const int n0 = tn * S::kTN, m0 = tm * S::kTM;
  constexpr int kHalf = S::kLaneN / 2;
  tile::Copies<S> at;
  tile::copy_offsets<S>(at, g.k, g.k, [&](int r) {
    if constexpr (EPI != PP_SILU) return r;
    const int j = r % S::kLaneN;
    return (j < kHalf ? 0 : g.n / 2) + (r / S::kLaneN) * kHalf + j % kHalf;
  });
  tile::Acc<S> acc;
  acc.zero();
  const int first = EPI == PP_SILU ? n0 / 2 : n0;
  tile::product<S>(sh, g.a + (size_t)m0 * g.k, (uint32_t)min(S::kTM, g.rows - m0) * g.k * 2, g.w + (size_t)first * g.k,
                   (uint32_t)(g.n - first) * g.k * 2, at, g.k / tile::kStep, acc);
  tile::each_row<S>(acc, m0, n0, g.rows, [&](int m, int n, float (&v)[S::kLaneN]) {
    if constexpr (EPI == PP_SILU) {
      float f[kHalf];
#pragma unroll
      for (int i = 0; i < kHalf; ++i) {
        const float h = round_bf16(v[i]);
        f[i] = round_bf16(tile::over_one_plus_exp(h, h)) * round_bf16(v[kHalf + i]);
      }
      uint16_t* c = g.c + (size_t)m * g.ldc + n / 2;
      if constexpr (kHalf >= 4) {
        tile::store_bf16<kHalf>(c, f, true);
      } else {
        *reinterpret_cast<uint32_t*>(c) = pack_pair(f[0], f[1]);
      }
    } else {
      uint16_t* c = g.c + (size_t)m * g.ldc + n;
      if constexpr (EPI == PP_RESIDUAL) {
        float x[S::kLaneN];
        tile::load_bf16<S::kLaneN>(c, x);
#pragma unroll
        for (int i = 0; i < S::kLaneN; ++i) v[i] = x[i] + round_bf16(v[i]);
      }
      tile::store_bf16<S::kLaneN>(c, v, true);
    }
  });
}

template <int EPI>
void launch_gemm(PpGemm g, hipStream_t s) {
  tile::with_shape(g.rows, g.n, 1, [&](auto shape) {
    using S = decltype(shape);
    g.tiles = tile::tiles_of<S>(g.rows, g.n, (int64_t)g.rows * g.k * 2);
    const int blocks = ahead_blocks(g.ahead, g.tiles.blocks(), S::kThreads);
    k_pp_gemm<EPI, S><<<blocks, S::kThreads, sizeof(tile::Lds<S>), s>>>(g);
  });
}

// ------------------------------------------------------------------ conv gate

// y = the gated short conv of in_proj's rows [B | C | x] (big, 3072 wide):
// bx = bf16(B x), the window of the row's and the two earlier bx (the
// sequence's state before its run), conv_gate_channel's rounding points. A
// thread takes 8 channels of one row. The thread of a run's first row also
// takes its second, the only other one that reads the old state, and then
// leaves the last three bx as the new state: no other thread touches it.
__global__ void __launch_bounds__(256) k_pp_conv(Prompt p, int l, int ci) {
  constexpr int kCols = kHidden / 8;  // threads per row
  const int m = blockIdx.x * (256 / kCols) + threadIdx.x / kCols, c0 = 8 * (threadIdx.x % kCols);
  if (m >= p.rows) return;
  const Row r = p.table[m];
  if (r.chunk == 1) return;
  float tap[3][8];
  {
    const uint4* t = reinterpret_cast<const uint4*>(conv_tensor<C_CONVW>(p.weights, l) + c0 * kConvTaps);
    const uint4 q[3] = {t[0], t[1], t[2]};
    const uint16_t* u = reinterpret_cast<const uint16_t*>(q);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) tap[j][i] = bf16_to_f32(u[3 * i + j]);
  }
  const auto bx_of = [&](int row, float (&v)[8]) {
    const uint16_t* s = p.big + (size_t)row * 3 * kHidden + c0;
    float b[8], x[8];
    unpack8(load8(s), b);
    unpack8(load8(s + 2 * kHidden), x);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = round_bf16(b[i] * x[i]);
  };
  const auto gate = [&](int row, const float (&a)[8], const float (&b)[8], const float (&bx)[8]) {
    float c[8], o[8];
    unpack8(load8(p.big + (size_t)row * 3 * kHidden + kHidden + c0), c);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float p0 = round_bf16(a[i] * tap[0][i]), p1 = round_bf16(b[i] * tap[1][i]), p2 = round_bf16(bx[i] * tap[2][i]);
      o[i] = c[i] * round_bf16((p0 + p1) + p2);
    }
    tile::store_bf16<8>(p.y + (size_t)row * kHidden + c0, o, true);
  };
  float a[8], b[8], bx[8];
  if (r.chunk >= 2) {
    bx_of(m - 2, a);
    bx_of(m - 1, b);
    bx_of(m, bx);
    gate(m, a, b, bx);
    return;
  }
  uint16_t* state = p.conv_state + ((size_t)(r.seq * LFM25_CONV_LAYERS + ci) * kHidden + c0) * kConvTaps;
  uint16_t st[24];
#pragma unroll
  for (int i = 0; i < 24; ++i) st[i] = state[i];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    a[i] = bf16_to_f32(st[3 * i + 1]);
    b[i] = bf16_to_f32(st[3 * i + 2]);
  }
  bx_of(m, bx);
  gate(m, a, b, bx);
  float win[3][8];  // the last three bx of the run, older ones from the state
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    win[0][i] = a[i];
    win[1][i] = b[i];
    win[2][i] = bx[i];
  }
  if (r.to_end >= 1) {
    float bx1[8];
    bx_of(m + 1, bx1);
    gate(m + 1, b, bx, bx1);
    if (r.to_end >= 2) {
      bx_of(m + r.to_end - 2, win[0]);
    } else {  // a run of two rows: the state's last bx stays
#pragma unroll
      for (int i = 0; i < 8; ++i) win[0][i] = b[i];
    }
    bx_of(m + r.to_end - 1, win[1]);
    bx_of(m + r.to_end, win[2]);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) state[3 * i + j] = f32_to_bf16(win[j][i]);
}

// ------------------------------------------------------------------ attention

// QK-RMSNorm + RoPE of a row's queries (in place) and keys, keys and values
// appended to the row's sequence cache: one block per row of q|k|v (big, 2048
// wide), a thread per 8 dimensions, eight threads per head.
__global__ void __launch_bounds__(256) k_pp_qkv(Prompt p, int l, int att) {
  const int m = blockIdx.x, t = threadIdx.x;
  const Row r = p.table[m];
  uint16_t* src = p.big + (size_t)m * 2 * kHidden + 8 * t;
  const int head = t / 8, d0 = 8 * (t % 8);  // 0..15 q, 16..23 k, 24..31 v
  if (head >= 24) {
    *reinterpret_cast<uint4*>(p.value_cache + pp_kv_base(p, r.seq, att, head - 24) + (size_t)r.pos * kHeadDim + d0) =
        *reinterpret_cast<const uint4*>(src);
    return;
  }
  float v[8], g[8], cs[8], sn[8];
  unpack8(load8(src), v);
  unpack8(load8((head < 16 ? attn_tensor<A_QLN>(p.weights, l) : attn_tensor<A_KLN>(p.weights, l)) + d0), g);
  unpack8(load8(p.rope + (size_t)r.pos * 2 * kHeadDim + d0), cs);
  unpack8(load8(p.rope + (size_t)r.pos * 2 * kHeadDim + kHeadDim + d0), sn);
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) ss = fmaf(v[i], v[i], ss);
  ss = group_sum<8>(ss);
  const float sc = 1.0f / sqrtf(ss * (1.0f / (float)kHeadDim) + kNormEps);
  float o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = round_bf16(round_bf16(v[i] * sc) * g[i]);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float partner = __shfl_xor(v[i], 4, kWave);  // dimension d +- 32
    const float rot = d0 < 32 ? -partner : partner;
    o[i] = round_bf16(v[i] * cs[i]) + round_bf16(rot * sn[i]);
  }
  uint16_t* dst = head < 16 ? src : p.key_cache + pp_kv_base(p, r.seq, att, head - 16) + (size_t)r.pos * kHeadDim + d0;
  tile::store_bf16<8>(dst, o, true);
}

__device__ __forceinline__ float max_groups(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(c[0]), __uint_as_float(c[1]));
}
__device__ __forceinline__ float sum_groups(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(c[0]) + __uint_as_float(c[1]);
}

// Causal attention of kQ query positions of one run and one KV head: the two
// query heads' columns share every key and value tile. The eager form's numbers (s_j = bf16(q . k_j) * 0.125; p_j = bf16(e^(s_j - m)
// / z); ctx = bf16(sum_j p_j v_j)) need m and z before the first p, so the
// keys are passed twice: once for m and z, once for the context. A wave owns
// 16 columns (one head, 16 positions); keys are the products' rows, so a lane
// holds one query's scores at 4 keys in 16 and its statistics need other
// lanes once, after the first pass. Key and value tiles of 64 positions come
// straight from the cache through three LDS stages; the value product's first
// operand is read from the row-major tile with the transposing LDS read.
//
// What bounds it is the arithmetic around the products (round, maximum,
// exponential, sum: about 17 issue slots a score over both passes against 3
// in the matrix cores), so the exponential is 2^(s c - m c) with c = log2(e) /
// 8 in one fused multiply-add and one v_exp.
constexpr int kKeys = 64;      // positions per tile
constexpr int kAttStages = 3;
struct AttLds {
  uint4 k[kAttStages][kKeys * 8];
  uint4 v[kAttStages][kKeys * 8];
};
// The transposing reads of a wave's 32 keys x 64 dimensions (16 lanes' 4 x 16
// blocks; lo: keys 0 .. 15, hi: 16 .. 31) and the wait for them, as one
// statement: the compiler puts a wait for every outstanding copy in front of
// the builtin form.
typedef short s16x4 __attribute__((ext_vector_type(4)));
struct ValueReads {
  uint32_t a[4];
  __device__ __forceinline__ ValueReads operator+(uint32_t bytes) const {
    return ValueReads{{a[0] + bytes, a[1] + bytes, a[2] + bytes, a[3] + bytes}};
  }
};
__device__ __forceinline__ void read_values(const ValueReads& at, s16x4 (&lo)[4], s16x4 (&hi)[4]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\t"
      "ds_read_b64_tr_b16 %1, %9\n\t"
      "ds_read_b64_tr_b16 %2, %10\n\t"
      "ds_read_b64_tr_b16 %3, %11\n\t"
      "ds_read_b64_tr_b16 %4, %8 offset:2048\n\t"
      "ds_read_b64_tr_b16 %5, %9 offset:2048\n\t"
      "ds_read_b64_tr_b16 %6, %10 offset:2048\n\t"
      "ds_read_b64_tr_b16 %7, %11 offset:2048\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(lo[0]), "=&v"(lo[1]), "=&v"(lo[2]), "=&v"(lo[3]), "=&v"(hi[0]), "=&v"(hi[1]), "=&v"(hi[2]), "=&v"(hi[3])
      : "v"(at.a[0]), "v"(at.a[1]), "v"(at.a[2]), "v"(at.a[3])
      : "memory");
}

template <int kQ>
__global__ void __launch_bounds__(kQ * 8) k_pp_attention(Prompt p, PromptRuns runs, int att) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host pass has no LDS address space)
  constexpr int kWaves = kQ / 8, kCopies = 8 / kWaves;  // copy instructions per wave and 64-row tile
  __shared__ AttLds sh;
  // This block's KV head and query tile. Tiles cost by their position, and up
  // to about two blocks land on a CU, block i and block i + 256: the first
  // half of the blocks takes the tiles from the longest down, the second half
  // the rest from the shortest up, so that a CU's two add up to the same
  // (3,900 rows: 151 -> 113 us; with the heads apart in the grid a CU could
  // get two of the longest). Consecutive blocks are the eight heads, so an
  // XCD reads one head's keys and values at a time.
  const int half = gridDim.x / (2 * kKvHeads) * kKvHeads, i = blockIdx.x;
  const int rank = i < half ? i : (int)gridDim.x - 1 - (i - half);
  const int g = rank % kKvHeads;
  int r = 0, first = 0, tile_at = rank / kKvHeads;
  while (true) {
    const int tiles = (runs.run[r].count + kQ - 1) / kQ;
    if (tile_at < tiles) {
      tile_at = tiles - 1 - tile_at;
      break;
    }
    tile_at -= tiles;
    first += runs.run[r++].count;
  }
  const int count = runs.run[r].count, pos0 = runs.run[r].position, seq = runs.run[r].sequence;
  const int w = wave_id(), l = lane_id();
  const int q0 = tile_at * kQ;                              // the block's first query within the run
  const int end = pos0 + min(q0 + kQ, count);               // cached positions any of its queries sees
  const int tiles = (end + kKeys - 1) / kKeys;
  const size_t base = pp_kv_base(p, seq, att, g);
  // this wave's columns: query head 2g + w % 2, positions 16 (w / 2) .. + 15
  const int qi = q0 + 16 * (w / 2) + (l & 15);              // this lane's query within the run
  const int pos = pos0 + qi;
  const int row = first + min(qi, count - 1);
  bf16x8 q[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    q[h] = __builtin_bit_cast(bf16x8, load8(p.big + (size_t)row * 2 * kHidden + (2 * g + w % 2) * kHeadDim + 32 * h + 8 * (l >> 4)));
  int off[kCopies];
#pragma unroll
  for (int i = 0; i < kCopies; ++i) {
    const int slot = (kCopies * w + i) * kWave + l, kr = slot / 8, c = (slot % 8) ^ tile::a_swizzle(kr);
    off[i] = (kr * kHeadDim + 8 * c) * 2;
  }
  // keys (and values) of tile t. Rows past the last seen position repeat that
  // position's: their weight is 0, and 0 times whatever lies there might be a
  // NaN. Tiles past it load nothing and are not read.
  const auto copy = [&](int t, int stage, bool values) {
    const int left = max(end - t * kKeys, 0);
    const uint32_t bytes = (uint32_t)min(left, kKeys) * kHeadDim * 2;
    const size_t at = base + (left > 0 ? (size_t)t * kKeys * kHeadDim : 0);
    const tile::Rsrc rk = tile::make_rsrc(p.key_cache + at, bytes), rv = tile::make_rsrc(p.value_cache + at, bytes);
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {
      const int o = min(off[i], (left - 1) * kHeadDim * 2 + (off[i] & (kHeadDim * 2 - 1)));
      tile::LdsVoid* dst = (tile::LdsVoid*)&sh.k[stage][(kCopies * w + i) * kWave];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, dst, 16, o, 0, 0, 0);
    }
    if (values) {
#pragma unroll
      for (int i = 0; i < kCopies; ++i) {
        const int o = min(off[i], (left - 1) * kHeadDim * 2 + (off[i] & (kHeadDim * 2 - 1)));
        tile::LdsVoid* dst = (tile::LdsVoid*)&sh.v[stage][(kCopies * w + i) * kWave];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, dst, 16, o, 0, 0, 0);
      }
    }
  };
  constexpr float kC = 0.125f * 1.44269504088896340736f;
  // The exponent of a score s is s kc - mc, kc = kC and mc = m kC rounded for
  // the maximum m. What the rounding leaves at s = m is in the sum and in
  // every probability alike; that it stays in exp2's range too, m kc ends at
  // kLarge kC (then it is at most 2^3, and the next smaller BF16 score is
  // still 2^19 below in the exponent). A lane that has seen no key has m =
  // kNone, below every score.
  constexpr float kLarge = 0x1p30f, kNone = -0x1.fffffep127f;
  const auto reference = [&](float m, float& kc, float& mc) {
    const float a = fabsf(m);
    kc = a > kLarge ? kC * kLarge / a : kC;
    mc = m * kc;
  };
  // What a sum formed with (m, mc) is scaled by to continue with (to, mc_to):
  // with maxima 2^22 apart nothing of it is left, and nearer ones have the same kc.
  const auto rescale = [&](float m, float mc, float to, float mc_to) {
    return to - m >= 0x1p22f ? 0.0f : __builtin_amdgcn_exp2f(mc - mc_to);
  };
  // scores of tile t: s[kt][e] = bf16(q . k) of key 64 t + 16 kt + 4 (l / 16) + e
  f32x4 s[4];
  const auto scores = [&](int t, int stage) {
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      s[kt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      const int kr = 16 * kt + (l & 15);
#pragma unroll
      for (int h = 0; h < 2; ++h)
        s[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8, sh.k[stage][kr * 8 + ((4 * h + (l >> 4)) ^ tile::a_swizzle(kr))]), q[h], s[kt], 0, 0, 0);
    }
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        const uint32_t b = pack_pair(s[kt][e], s[kt][e + 1]);
        s[kt][e] = lo_f32(b);
        s[kt][e + 1] = hi_f32(b);
      }
    if (t * kKeys + kKeys - 1 > pos0 + q0) {  // a tile that some query does not see whole
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (t * kKeys + 16 * kt + 4 * (l >> 4) + e > pos) s[kt][e] = -INFINITY;
    }
  };
  // tile t's copies (kN of them per tile and wave) have landed, in every
  // wave; the stage that tile t - 1 was read from is free
#define LFM25_PP_WAIT(kN) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kN) : "memory")
  copy(0, 0, false);
  copy(1, 1, false);
  // m: this lane's largest score so far, z: the sum of 2^(s kc - mc), scaled
  // by the difference of the rounded mc that its terms were and will be formed
  // with. (Scaled by 2^(m kC - mc), which is not 1 where m did not change, it
  // was up to 4e-5 off after 64 tiles.)
  float m = kNone, kc, mc, z = 0.0f;
  reference(m, kc, mc);
  int stage = 0;
  for (int t = 0; t < tiles; ++t) {
    LFM25_PP_WAIT(kCopies);
    copy(t + 2, stage == 0 ? 2 : stage - 1, false);
    scores(t, stage);
    float top = s[0][0];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) top = fmaxf(top, s[kt][e]);
    const float to = fmaxf(m, top), mc0 = mc;
    kc = kC;
    mc = to * kC;
    float f = __builtin_amdgcn_exp2f(mc0 - mc);
    if (__builtin_amdgcn_ballot_w64(to > kLarge || m < -kLarge) != 0) {  // (rare past the first tile)
      reference(to, kc, mc);
      f = rescale(m, mc0, to, mc);
    }
    m = to;
    float sum = 0.0f;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) sum += __builtin_amdgcn_exp2f(fmaf(s[kt][e], kc, -mc));
    z = fmaf(z, f, sum);
    stage = stage == 2 ? 0 : stage + 1;
  }
  {
    const float all = max_groups(m), mc0 = mc;
    reference(all, kc, mc);
    z = sum_groups(z * rescale(m, mc0, all, mc));
  }
  const float rz = 1.0f / z;
  // LDS addresses of this lane's value reads: row 4 (l / 16) + (l % 16) / 4 of
  // 16, 8 bytes at dimensions 16 dt + 4 (l % 4) (rows 16 apart keep a_swizzle)
  ValueReads at;
  {
    const int vr = 4 * (l >> 4) + (l & 15) / 4;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
      at.a[dt] = (uint32_t)(uintptr_t)(tile::LdsVoid*)&sh.v[0][vr * 8 + ((2 * dt + (l & 3) / 2) ^ tile::a_swizzle(vr))] + 8 * (l & 1);
  }
  f32x4 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  LFM25_PP_WAIT(0);  // the first pass's copies and reads
  copy(0, 0, true);
  copy(1, 1, true);
  stage = 0;
  for (int t = 0; t < tiles; ++t) {
    LFM25_PP_WAIT(2 * kCopies);
    copy(t + 2, stage == 0 ? 2 : stage - 1, true);
    scores(t, stage);
#pragma unroll
    for (int c = 0; c < 2; ++c) {  // 32 keys: a lane's 4 of key tile 2c, then its 4 of 2c + 1
      uint32_t pw[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4& sk = s[2 * c + i / 2];
        pw[i] = pack_pair(__builtin_amdgcn_exp2f(fmaf(sk[2 * (i % 2)], kc, -mc)) * rz,
                      __builtin_amdgcn_exp2f(fmaf(sk[2 * (i % 2) + 1], kc, -mc)) * rz);
      }
      const bf16x8 pf = __builtin_bit_cast(bf16x8, uint4{pw[0], pw[1], pw[2], pw[3]});
      s16x4 v0[4], v1[4];  // V^T: dimension 16 dt + l % 16 of those 8 keys
      read_values(at + stage * (kKeys * kHeadDim * 2) + c * (32 * kHeadDim * 2), v0, v1);
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8, __builtin_shufflevector(v0[dt], v1[dt], 0, 1, 2, 3, 4, 5, 6, 7)), pf, o[dt], 0, 0, 0);
    }
    stage = stage == 2 ? 0 : stage + 1;
  }
#undef LFM25_PP_WAIT
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // before the block's LDS is given back
  if (qi >= count) return;
  // o[dt]: dimensions 16 dt + 4 (l / 16) + e of this lane's query
  uint16_t* dst = p.y + (size_t)row * kHidden + (2 * g + w % 2) * kHeadDim + 4 * (l >> 4);
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
    *reinterpret_cast<uint2*>(dst + 16 * dt) = uint2{pack_pair(o[dt][0], o[dt][1]), pack_pair(o[dt][2], o[dt][3])};
#endif
}

template <int kQ>
void launch_attention(const Prompt& p, const PromptRuns& runs, int att, hipStream_t s) {
  int tiles = 0;
  for (int r = 0; r < runs.n; ++r) tiles += (runs.run[r].count + kQ - 1) / kQ;
  k_pp_attention<kQ><<<tiles * kKvHeads, kQ * 8, 0, s>>>(p, runs, att);
}

}  // namespace

size_t prompt_bytes(int rows) { return (size_t)rows * kPpRowBytes; }

int prompt_layers(const lfm25_batch* b, const int32_t* tokens, const PromptRuns& runs, void* ws, int32_t* status,
                  const uint16_t** x, hipStream_t s) {
  int rows = 0;
  for (int r = 0; r < runs.n; ++r) rows += runs.run[r].count;
  Prompt p{};
  p.weights = b->weights;
  p.embedding = b->embedding;
  p.rope = b->rope;
  p.conv_state = b->conv_state;
  p.key_cache = b->key_cache;
  p.value_cache = b->value_cache;
  p.x = static_cast<uint16_t*>(ws);
  p.xn = p.x + (size_t)rows * kHidden;
  p.y = p.xn + (size_t)rows * kHidden;
  p.big = p.y + (size_t)rows * kHidden;
  p.table = reinterpret_cast<Row*>(p.big + (size_t)rows * 3 * kHidden);
  p.status = status;
  p.rows = rows;
  p.capacity = b->capacity;
  p.vocab = b->vocab;
  const int norm_blocks = (rows + kNormRows - 1) / kNormRows;
  // the n x k weights w of a product to come
  const auto ahead = [&](const uint16_t* w, int n, int k, bool silu) {
    const int group = tile::ahead_group(rows, n, 1, (int64_t)rows * k * 2) / (silu ? 2 : 1);
    return Ahead{w, group > 0 ? n : 0, k / 64, group > 0 ? group : 1};
  };
  k_pp_embed<<<norm_blocks, kNormRows * kWave, 0, s>>>(p, runs, tokens);
  for (int l = 0; l < kLayers; ++l) {
    const bool attn = is_attn(l), next = is_attn(l + 1);
    const uint16_t *w = p.weights + layer_off(l), *nw = p.weights + layer_off(l + 1);
    const auto tensor = [&](int a, int c) { return w + slot_off(attn, attn ? a : c); };
    const uint16_t *w_out = tensor(A_O, C_OUT), *w_up = tensor(A_W1, C_W1), *w_down = tensor(A_W2, C_W2);
    const Ahead out = ahead(w_out, kHidden, kHidden, false), up = ahead(w_up, 2 * kFfn, kHidden, true);
    const Ahead down = ahead(w_down, kHidden, kFfn, false);
    const Ahead mixer = l + 1 == kLayers ? Ahead{nullptr, 0, 1, 1}
                        : ahead(nw + slot_off(next, next ? (int)A_Q : (int)C_IN), next ? 2 * kHidden : 3 * kHidden, kHidden, false);
    if (attn) {
      const int att = l - conv_before(l);
      launch_gemm<PP_STORE>(PpGemm{p.xn, tensor(A_Q, 0), p.big, rows, 2 * kHidden, kHidden, 2 * kHidden, {}, {{out, up}, 0}}, s);
      k_pp_qkv<<<rows, 256, 0, s>>>(p, l, att);
      // query positions per block: as many as still leave a block per CU
      if (rows >= 32 * 64) launch_attention<64>(p, runs, att, s);
      else if (rows >= 32 * 32) launch_attention<32>(p, runs, att, s);
      else launch_attention<16>(p, runs, att, s);
    } else {
      launch_gemm<PP_STORE>(PpGemm{p.xn, tensor(0, C_IN), p.big, rows, 3 * kHidden, kHidden, 3 * kHidden, {}, {{out, up}, 0}}, s);
      k_pp_conv<<<(rows + 1) / 2, 256, 0, s>>>(p, l, conv_before(l));
    }
    launch_gemm<PP_RESIDUAL>(PpGemm{p.y, w_out, p.x, rows, kHidden, kHidden, kHidden, {}, {}}, s);
    k_pp_norm<<<norm_blocks, kNormRows * kWave, 0, s>>>(p.x, tensor(A_FFNNORM, C_FFNNORM), p.xn, rows);
    launch_gemm<PP_SILU>(PpGemm{p.xn, w_up, p.big, rows, 2 * kFfn, kHidden, kFfn, {}, {{down, mixer}, 0}}, s);
    launch_gemm<PP_RESIDUAL>(PpGemm{p.big, w_down, p.x, rows, kHidden, kFfn, kHidden, {}, {}}, s);
    if (l + 1 < kLayers)
      k_pp_norm<<<norm_blocks, kNormRows * kWave, 0, s>>>(
          p.x, nw + slot_off(next, next ? (int)A_OPNORM : (int)C_OPNORM), p.xn, rows);
  }
  *x = p.x;
  return check_launch("prompt pass");
}

}  // namespace lfm25
