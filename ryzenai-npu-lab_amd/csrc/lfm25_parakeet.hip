// Parakeet (FastConformer) encoder on gfx950: the reference's all-NPU encoder
// (experiments/pk_model.py, pk_engine.py, kernels/pk/pk_core.cc, pk_fast.cc)
// as four kernels per block phase kind, one stream:
//
//   GEMM      C = bf16(epi(A . B + bias)) on the matrix cores, 32 x 64 to
//             256 x 128 block tiles (lfm25_gemm.h; replaces gemm_step / pk_wx /
//             epilogue, pk_fast.cc:167-231, pk_core.cc:169-183)
//   LN        scaled residual + LayerNorm (+ a second LayerNorm)
//             (layer_norm / residual / ln_frame, pk_core.cc:55-116)
//   ATT       relative-position attention of one (sequence, head)
//             (att_queries / att_bd / att_keys / att_finish,
//             pk_core.cc:126-203, pk_fast.cc:71-116)
//   CONV      GLU + 9-tap depthwise conv + bias + Swish (conv_frames,
//             pk_fast.cc:119-154)
//
// and the 22-phase block order of build_phases (pk_model.py:132-161) on the
// host. Rounding points are those of the reference's BF16 mirror
// (experiments/012_layer_test.py:45-114): FP32 inside a phase, BF16 where the
// NPU stores a field. Weight matrices are stored output-major ([out x in],
// every row contiguous in the reduction dimension) so both GEMM operands are
// read as 16-byte runs along K.
#include <algorithm>
#include <cstring>
#include <vector>

#include "lfm25_host.h"
#include "lfm25_ahead.h"
#include "lfm25_device.h"
#include "lfm25_gemm.h"

namespace lfm25 {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kD = 1024;
constexpr int kPkHeads = 8;
constexpr int kDk = 128;
constexpr int kPkFfn = 4096;
constexpr int kConvTapsPk = 9;
constexpr float kLnEps = 1.0e-5f;

// Sum / maximum over the four lanes l, l ^ 16, l ^ 32, l ^ 48 (gfx950 row swaps).
__device__ __forceinline__ float sum_lanes16(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(c[0]) + __uint_as_float(c[1]);
}
__device__ __forceinline__ float max_lanes16(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(c[0]), __uint_as_float(c[1]));
}

// ------------------------------------------------------------------ GEMM

// C[m][n] = bf16(epi(sum_k A[m][k] Bt[n][k] + bias[n])), one block tile per
// block (lfm25_gemm.h; blockIdx.x: tile, blockIdx.y: K split). EPI_RESIDUAL:
// C = bf16(C + scale bf16(sum)), C the residual stream.
//
// Split K (kSplit): block z covers K range [z * kchunk, (z + 1) * kchunk) and
// writes its FP32 partial tile to part[z][M][N]; k_pk_splitk or
// k_pk_reduce_ln sums the splits in index order and applies the epilogue, so
// the result does not depend on which blocks ran when.
constexpr int kBN = 128;          // n is a multiple of this
constexpr int kBK = tile::kStep;  // and k of this
constexpr int kMinChunk = 512;    // smallest K range of a split
enum PkEpi { EPI_NONE = 0, EPI_BIAS = 1, EPI_SWISH = 2, EPI_RESIDUAL = 3 };

struct PkGemm {
  const uint16_t* A;
  const uint16_t* Bt;
  const uint16_t* bias;
  uint16_t* C;
  float* part;
  float scale;  // EPI_RESIDUAL
  int lda, ldb, ldc, M, N, kchunk;
  bool wide;    // C and its rows are 16-byte aligned
  tile::Tiles tiles;
  AheadPair ahead;  // weights of the products to come (unsplit products only)
};

template <int EPI>
__device__ __forceinline__ float epilogue(float v, float b) {
  if (EPI == EPI_BIAS) v = v + b;
  if (EPI == EPI_SWISH) v = tile::over_one_plus_exp(v, v);
  return v;
}

template <int EPI, bool kSplit, bool kFar, typename S>
__global__ void __launch_bounds__(S::kThreads, 2) k_pk_gemm(const PkGemm g) {
  extern __shared__ __attribute__((aligned(16))) char lds_raw[];
  auto& sh = *reinterpret_cast<tile::Lds<S>*>(lds_raw);
  const int own = g.tiles.blocks();
  if (!kSplit && (int)blockIdx.x >= own) return read_ahead(g.ahead, own);
  int tm, tn;
  if (!g.tiles.of(blockIdx.x, tm, tn)) return;
  const int n0 = tn * S::kTN, m0 = tm * S::kTM, z = blockIdx.y;
  const size_t kbeg = kSplit ? (size_t)z * g.kchunk : 0;
  tile::Copies<S> at;
  tile::Acc<S> acc;
  if constexpr (kFar) {
    const tile::FarRows<S> far(g.A + (size_t)m0 * g.lda + kbeg, g.lda, min(S::kTM, g.M - m0),
                               g.Bt + (size_t)n0 * g.ldb + kbeg, g.ldb);
    acc.zero();
    tile::product<S, true>(sh, nullptr, 0, nullptr, 0, at, g.kchunk / kBK, acc, &far);
  } else {
    tile::copy_offsets<S>(at, g.lda, g.ldb, [](int r) { return r; });
    acc.zero();
    // a descriptor ends with the last row's last K element of this block's range
    tile::product<S>(sh, g.A + (size_t)m0 * g.lda + kbeg,
                     ((uint32_t)(min(S::kTM, g.M - m0) - 1) * g.lda + g.kchunk) * 2, g.Bt + (size_t)n0 * g.ldb + kbeg,
                     ((uint32_t)(S::kTN - 1) * g.ldb + g.kchunk) * 2, at, g.kchunk / kBK, acc);
  }
  tile::each_row<S>(acc, m0, n0, g.M, [&](int m, int n, float (&v)[S::kLaneN]) {
    if constexpr (kSplit) {
      f32x4_t* p = reinterpret_cast<f32x4_t*>(g.part + ((size_t)z * g.M + m) * g.N + n);
#pragma unroll
      for (int i = 0; i < S::kLaneN / 4; ++i) p[i] = f32x4_t{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
    } else {
      uint16_t* c = g.C + (size_t)m * g.ldc + n;
      if constexpr (EPI == EPI_RESIDUAL) {
        float x[S::kLaneN];
        tile::load_bf16<S::kLaneN>(c, x);
#pragma unroll
        for (int i = 0; i < S::kLaneN; ++i) v[i] = x[i] + g.scale * round_bf16(v[i]);
      } else {
#pragma unroll
        for (int i = 0; i < S::kLaneN; ++i) v[i] = epilogue<EPI>(v[i], EPI == EPI_BIAS ? bf16_to_f32(g.bias[n + i]) : 0.0f);
      }
      tile::store_bf16<S::kLaneN>(c, v, g.wide);
    }
  });
}

// y += partials z .. z + G - 1 of a thread's NQ x 4 values (partial i at
// p + i * stride), those below `splits` only, added in index order after all
// G loads are issued; a load past the last partial repeats the last one.
template <int G, int NQ>
__device__ __forceinline__ void add_partials(f32x4_t (&y)[NQ], const float* p, size_t stride, int z, int splits) {
  f32x4_t t[G][NQ];
#pragma unroll
  for (int u = 0; u < G; ++u) {
    const int zu = z + u < splits ? z + u : splits - 1;
#pragma unroll
    for (int q = 0; q < NQ; ++q) t[u][q] = *reinterpret_cast<const f32x4_t*>(p + zu * stride + 4 * q);
  }
  __builtin_amdgcn_sched_barrier(0);  // every load issued before the first wait
#pragma unroll
  for (int u = 0; u < G; ++u)
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const f32x4_t r = f32x4_t{y[q][0] + t[u][q][0], y[q][1] + t[u][q][1], y[q][2] + t[u][q][2],
                                y[q][3] + t[u][q][3]};
      y[q] = z + u < splits ? r : y[q];
    }
}
// y = the sum of partials 0 .. splits - 1 in index order, from -0 (x + -0 is
// x for every x, the sign of zero included), G partials' loads in flight per
// round trip. The host picks G from the split count (partial_group): one
// straight-line group per round trip, with no branch for the compiler to
// hoist a shared first load out of.
template <int G, int NQ>
__device__ __forceinline__ void sum_partials(f32x4_t (&y)[NQ], const float* p, size_t stride, int splits) {
#pragma unroll
  for (int q = 0; q < NQ; ++q) y[q] = f32x4_t{-0.0f, -0.0f, -0.0f, -0.0f};
  for (int z = 0; z < splits; z += G) add_partials<G>(y, p, stride, z, splits);
}
// Partials per round trip for `splits` of them: the next power of two, at
// most 8 (lfm25_pk_gemm's callers name any; the encoder's have 2 or 4).
inline int partial_group(int splits) { return splits <= 1 ? 1 : splits <= 2 ? 2 : splits <= 4 ? 4 : 8; }

// Sum of the `splits` FP32 partial products in index order (G of them per
// round trip), epilogue, BF16: one thread per four consecutive outputs of
// row blockIdx.x (blockIdx.y: the row's 1024-wide column range).
template <int EPI, int G>
__global__ void __launch_bounds__(256) k_pk_splitk(const float* __restrict__ part, int splits, int M, int N,
                                                   const uint16_t* __restrict__ bias, uint16_t* __restrict__ C,
                                                   int ldc) {
  const int m = blockIdx.x, n = 4 * (blockIdx.y * 256 + threadIdx.x);
  if (n >= N) return;
  float bs[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // loaded first: in flight with the partials
  if (EPI == EPI_BIAS) {
#pragma unroll
    for (int e = 0; e < 4; ++e) bs[e] = bf16_to_f32(bias[n + e]);
  }
  f32x4_t v[1];
  sum_partials<G>(v, part + (size_t)m * N + n, (size_t)M * N, splits);
  u32x2_t pk;
  pk.x = (uint32_t)f32_to_bf16(epilogue<EPI>(v[0][0], bs[0])) |
         ((uint32_t)f32_to_bf16(epilogue<EPI>(v[0][1], bs[1])) << 16);
  pk.y = (uint32_t)f32_to_bf16(epilogue<EPI>(v[0][2], bs[2])) |
         ((uint32_t)f32_to_bf16(epilogue<EPI>(v[0][3], bs[3])) << 16);
  *reinterpret_cast<u32x2_t*>(C + (size_t)m * ldc + n) = pk;
}

// ------------------------------------------------------------------ LayerNorm

// A lane's 16 BF16 values as loaded (two 16-byte words): unpacked where used,
// so a load issued early is not waited for until then.
struct Row16 {
  uint4 a, b;
};
__device__ __forceinline__ Row16 load_raw16(const uint16_t* p) {
  const uint4* q = reinterpret_cast<const uint4*>(p);
  return Row16{q[0], q[1]};
}
__device__ __forceinline__ void unpack16(const Row16& r, float* v) {
  const uint32_t w[8] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    v[2 * i] = lo_f32(w[i]);
    v[2 * i + 1] = hi_f32(w[i]);
  }
}
__device__ __forceinline__ void load_row16(const uint16_t* p, float* v) { unpack16(load_raw16(p), v); }
__device__ __forceinline__ void store_row16(uint16_t* p, const float* v) {
  uint32_t w[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) w[i] = (uint32_t)f32_to_bf16(v[2 * i]) | ((uint32_t)f32_to_bf16(v[2 * i + 1]) << 16);
  uint4* q = reinterpret_cast<uint4*>(p);
  q[0] = uint4{w[0], w[1], w[2], w[3]};
  q[1] = uint4{w[4], w[5], w[6], w[7]};
}

// bf16((v - mean) / sqrt(var + eps) * g + b) of one 1024-row held 16 per lane
// (lane l: elements 16l .. 16l + 15); mean and variance in FP32 (wave sums).
// g / b: the lane's 16 gammas and betas.
__device__ __forceinline__ void ln_apply(const float* v, const Row16& g, const Row16& b, float* out) {
  float gv[16], bv[16];
  unpack16(g, gv);
  unpack16(b, bv);
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i) s += v[i];
  const float mu = wave_sum(s) * (1.0f / (float)kD);
  float q = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float d = v[i] - mu;
    q += d * d;
  }
  const float var = wave_sum(q) * (1.0f / (float)kD);
  const float den = sqrtf(var + kLnEps);
#pragma unroll
  for (int i = 0; i < 16; ++i) out[i] = round_bf16((v[i] - mu) / den * gv[i] + bv[i]);
}

// A lane's 16 gammas and betas of LN1 and, when g2 is given, of LN2: loaded
// before the row they norm is formed, so their loads overlap the row's.
struct LnLane {
  Row16 g1, b1, g2, b2;
  bool two;
};
__device__ __forceinline__ void load_ln(LnLane& p, const uint16_t* g1, const uint16_t* b1, const uint16_t* g2,
                                        const uint16_t* b2) {
  p.g1 = load_raw16(g1 + 16 * lane_id());
  p.b1 = load_raw16(b1 + 16 * lane_id());
  p.two = g2 != nullptr;
  if (p.two) {
    p.g2 = load_raw16(g2 + 16 * lane_id());
    p.b2 = load_raw16(b2 + 16 * lane_id());
  }
}

// The norm modes of one row m given x' (v, 16 per lane). "carry"
// (normed_x == 0): x <- x' when store_x, a <- LN1(x'). "normed"
// (normed_x == 1): x <- LN1(x') and, when LN2 is given, a <- LN2(x)
// (ln_frame's DOUBLE/FINAL, pk_core.cc:99-116).
__device__ __forceinline__ void ln_modes(uint16_t* x, int m, const float* v, bool store_x, const LnLane& p,
                                         int normed_x, uint16_t* a) {
  const size_t off = (size_t)m * kD + 16 * lane_id();
  float o[16];
  ln_apply(v, p.g1, p.b1, o);
  if (!normed_x) {
    if (store_x) store_row16(x + off, v);
    store_row16(a + off, o);
    return;
  }
  store_row16(x + off, o);
  if (p.two) {
    float o2[16];
    ln_apply(o, p.g2, p.b2, o2);
    store_row16(a + off, o2);
  }
}

// One wave per row (four rows per block). x' = y ? bf16(x + s * y) : x, then
// ln_modes.
constexpr int kLnRows = 4;
__global__ void __launch_bounds__(kLnRows* kWave) k_pk_ln(uint16_t* __restrict__ x, const uint16_t* __restrict__ y,
                                                          float s, const uint16_t* __restrict__ g1,
                                                          const uint16_t* __restrict__ b1,
                                                          const uint16_t* __restrict__ g2,
                                                          const uint16_t* __restrict__ b2, int normed_x,
                                                          uint16_t* __restrict__ a, int rows) {
  const int m = blockIdx.x * kLnRows + wave_id();
  if (m >= rows) return;
  const size_t off = (size_t)m * kD + 16 * lane_id();
  LnLane p;
  load_ln(p, g1, b1, g2, b2);
  float v[16];
  load_row16(x + off, v);
  if (y != nullptr) {
    float yv[16];
    load_row16(y + off, yv);
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = round_bf16(v[i] + s * yv[i]);
  }
  ln_modes(x, m, v, y != nullptr, p, normed_x, a);
}

// The end of a d-wide product whose `splits` FP32 partials sit in
// part[z][rows][1024]: y = bf16(sum of the partials in index order), then
// x' = bf16(x + s * y) and ln_modes (the GEMM's store, residual and
// LayerNorm phases of pk_core.cc:90-116 in one pass over the row). One row
// (wave) per block: only products of few rows are split, and a row's splits
// x 4 KB of partials are then spread over as many CUs as there are rows (a
// CU's load rate, not HBM, bounds this pass).
template <int G>
__global__ void __launch_bounds__(kWave) k_pk_reduce_ln(const float* __restrict__ part, int splits,
                                                                 uint16_t* __restrict__ x, float s,
                                                                 const uint16_t* __restrict__ g1,
                                                                 const uint16_t* __restrict__ b1,
                                                                 const uint16_t* __restrict__ g2,
                                                                 const uint16_t* __restrict__ b2, int normed_x,
                                                                 uint16_t* __restrict__ a, int rows) {
  const int m = blockIdx.x;
  const size_t off = (size_t)m * kD + 16 * lane_id();
  const size_t stride = (size_t)rows * kD;
  // the residual row and the norms' parameters first: in flight with the partials
  LnLane p;
  load_ln(p, g1, b1, g2, b2);
  const Row16 xr = load_raw16(x + off);
  f32x4_t y[4];
  sum_partials<G>(y, part + off, stride, splits);
  float v[16];
  unpack16(xr, v);
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = round_bf16(v[i] + s * round_bf16(y[i / 4][i % 4]));
  ln_modes(x, m, v, true, p, normed_x, a);
}

// ------------------------------------------------------------------ attention

// Relative-position attention of sequence b (blockIdx.y), head h
// (blockIdx.x) over T = 128 frames, `valid` of them real (keys j >= valid
// masked), as the mirror computes it (012_layer_test.py:67-86):
//   bd_ij' = bf16(q_i . P_h[:, j'])            (j' < 2T, position scores)
//   qu = bf16(q + delta_h); s_ij = qu_i . k_j + bd_i,T-1-i+j;
//   p = softmax_j(s) in FP32; o_i = bf16(sum_j p_ij v_j).
// q (scaled, bias_v folded in), k, v come from the q|k|v rows [T x 3072];
// P_h^T is the head's [2T x 128] position table (last row zero).
//
// Two ways to split the work (launch_attention chooses).
//
// k_pk_attention: two blocks per (sequence, head).
// The block first requests everything it reads (P, K and V into LDS, each
// wave's 16 query rows into registers) in one round of 16-byte loads. Each
// wave then forms its queries' position scores and key scores from LDS on
// the matrix cores (BF16 operands, exact products, FP32 sums); after a
// barrier the position scores go to LDS as BF16 over the P region, so the
// shifted index T-1-i+j can be read per element. The probabilities stay FP32
// through the value product by splitting each into a BF16 high part and a
// BF16 remainder (two MFMA chains); V^T is the first operand, so a lane's four
// results are four consecutive dimensions of one query (one 8-byte store).
constexpr int kAttT = 128;
constexpr int kAttWaves = 8;
constexpr int kQT = kAttT / 16 / kAttWaves;  // 16-query tiles per wave: 1
constexpr int kAttThreads = kAttWaves * kWave;
constexpr int kAttRow = kDk + 8;           // bf16 per LDS row of P, K, V^T (272 bytes: conflict-free 16-byte reads)
constexpr int kBdRow = 2 * kAttT + 8;      // bf16 per LDS row of the position scores
// V^T rows of 130 bf16 (65 words: consecutive rows start one bank apart), so
// the transposing 2-byte stores of 16 dimensions at one key spread over the
// banks; the rows are 4-byte aligned, so the operand reads are 4-byte.
constexpr int kVtRow = kAttT + 2;
struct PkAttLds {
  union {
    uint16_t p[2 * kAttT][kAttRow];        // P_h^T [j'][d] while the position scores are formed
    uint16_t bd[kAttT][kBdRow];            // then the BF16 position scores [i][j']
  } u;
  uint16_t k[kAttT][kAttRow];              // K [j][d]
  uint16_t vt[kDk][kVtRow];                // V^T [d][j]
};

__device__ __forceinline__ bf16x8_t as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8_t, v); }
__device__ __forceinline__ bf16x8_t lds_frag(const uint16_t* row, int col) {
  return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(row + col));
}

// kAttSplit blocks per (sequence, head), blockIdx.z taking query tiles
// [kAttWaves / kAttSplit z, + kAttWaves / kAttSplit): each block stages the
// whole P, K and V^T but forms only its queries' products, so at one window
// the 8 heads run on 16 CUs instead of 8.
constexpr int kAttSplit = 2;
constexpr int kAttBlockThreads = kAttThreads / kAttSplit;
__global__ void __launch_bounds__(kAttBlockThreads, 1)
    k_pk_attention(const uint16_t* __restrict__ qkv, const uint16_t* __restrict__ pos,
                   const uint16_t* __restrict__ delta, uint16_t* __restrict__ out, int valid) {
  __shared__ PkAttLds sh;
  const int h = blockIdx.x, b = blockIdx.y;
  // w: the wave's query tile (16 kQT w ..) over the (sequence, head)'s kAttWaves
  const int t = threadIdx.x, w = wave_id() + (kAttWaves / kAttSplit) * blockIdx.z, l = lane_id();
  const uint16_t* base = qkv + (size_t)b * kAttT * 3 * kD;
  const uint16_t* ph = pos + (size_t)h * 2 * kAttT * kDk;
  // one round of loads: P (16 chunks per thread), K and V (8 each), this wave's q fragments
  constexpr int kRowChunks16 = kDk / 8;  // 16-byte chunks per 128-wide row
  uint4 pr[2 * kAttT * kRowChunks16 / kAttBlockThreads], kr[kAttT * kRowChunks16 / kAttBlockThreads],
      vr[kAttT * kRowChunks16 / kAttBlockThreads];
#pragma unroll
  for (int i = 0; i < 2 * kAttT * kRowChunks16 / kAttBlockThreads; ++i) {
    const int c = t + kAttBlockThreads * i;
    pr[i] = *reinterpret_cast<const uint4*>(ph + (size_t)(c / kRowChunks16) * kDk + 8 * (c % kRowChunks16));
  }
#pragma unroll
  for (int i = 0; i < kAttT * kRowChunks16 / kAttBlockThreads; ++i) {
    const int c = t + kAttBlockThreads * i;
    const uint16_t* row = base + (size_t)(c / kRowChunks16) * 3 * kD + h * kDk + 8 * (c % kRowChunks16);
    kr[i] = *reinterpret_cast<const uint4*>(row + kD);
    vr[i] = *reinterpret_cast<const uint4*>(row + 2 * kD);
  }
  uint4 qraw[kQT][kDk / 32];  // query 16 kQT w + 16qt + l%16, dimensions 32ds + 8(l/16) .. + 7
#pragma unroll
  for (int qt = 0; qt < kQT; ++qt)
#pragma unroll
    for (int ds = 0; ds < kDk / 32; ++ds)
      qraw[qt][ds] = *reinterpret_cast<const uint4*>(base + (size_t)(16 * kQT * w + 16 * qt + (l & 15)) * 3 * kD +
                                                      h * kDk + 32 * ds + 8 * (l >> 4));
#pragma unroll
  for (int i = 0; i < 2 * kAttT * kRowChunks16 / kAttBlockThreads; ++i) {
    const int c = t + kAttBlockThreads * i;
    *reinterpret_cast<uint4*>(&sh.u.p[c / kRowChunks16][8 * (c % kRowChunks16)]) = pr[i];
  }
#pragma unroll
  for (int i = 0; i < kAttT * kRowChunks16 / kAttBlockThreads; ++i) {
    const int c = t + kAttBlockThreads * i;
    const int j = c / kRowChunks16, d0 = 8 * (c % kRowChunks16);
    *reinterpret_cast<uint4*>(&sh.k[j][d0]) = kr[i];
    const uint32_t vw[4] = {vr[i].x, vr[i].y, vr[i].z, vr[i].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sh.vt[d0 + 2 * e][j] = (uint16_t)(vw[e] & 0xffffu);
      sh.vt[d0 + 2 * e + 1][j] = (uint16_t)(vw[e] >> 16);
    }
  }
  lds_barrier();
  // position scores: bacc[pt][qt] lane holds j' = 16pt + 4(l/16) + e of query 16 kQT w + 16qt + l%16
  f32x4_t bacc[2 * kAttT / 16][kQT];
#pragma unroll
  for (int p = 0; p < 2 * kAttT / 16; ++p)
#pragma unroll
    for (int qt = 0; qt < kQT; ++qt) bacc[p][qt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int ds = 0; ds < kDk / 32; ++ds)
#pragma unroll
    for (int p = 0; p < 2 * kAttT / 16; ++p) {
      const bf16x8_t pf = lds_frag(sh.u.p[16 * p + (l & 15)], 32 * ds + 8 * (l >> 4));
#pragma unroll
      for (int qt = 0; qt < kQT; ++qt)
        bacc[p][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf, as_bf16x8(qraw[qt][ds]), bacc[p][qt], 0, 0, 0);
    }
  // key scores: acc[kt][qt] holds keys 16kt + 4(l/16) + e of query 16 kQT w + 16qt + l%16
  f32x4_t acc[8][kQT];
#pragma unroll
  for (int kt = 0; kt < 8; ++kt)
#pragma unroll
    for (int qt = 0; qt < kQT; ++qt) acc[kt][qt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int ds = 0; ds < kDk / 32; ++ds) {
    const int d0 = 32 * ds + 8 * (l >> 4);
    const uint4 dl = *reinterpret_cast<const uint4*>(delta + h * kDk + d0);
    const uint32_t dw[4] = {dl.x, dl.y, dl.z, dl.w};
    bf16x8_t qf[kQT];
#pragma unroll
    for (int qt = 0; qt < kQT; ++qt) {
      const uint32_t qw[4] = {qraw[qt][ds].x, qraw[qt][ds].y, qraw[qt][ds].z, qraw[qt][ds].w};
      uint32_t u[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        u[e] = (uint32_t)f32_to_bf16(lo_f32(qw[e]) + lo_f32(dw[e])) |
               ((uint32_t)f32_to_bf16(hi_f32(qw[e]) + hi_f32(dw[e])) << 16);
      qf[qt] = as_bf16x8(uint4{u[0], u[1], u[2], u[3]});
    }
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) {
      const bf16x8_t kf = lds_frag(sh.k[16 * kt + (l & 15)], d0);
#pragma unroll
      for (int qt = 0; qt < kQT; ++qt) acc[kt][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[qt], acc[kt][qt], 0, 0, 0);
    }
  }
  lds_barrier();  // every wave is done with P: its region takes the position scores
#pragma unroll
  for (int p = 0; p < 2 * kAttT / 16; ++p)
#pragma unroll
    for (int qt = 0; qt < kQT; ++qt) {
      u32x2_t pk;
      pk.x = (uint32_t)f32_to_bf16(bacc[p][qt][0]) | ((uint32_t)f32_to_bf16(bacc[p][qt][1]) << 16);
      pk.y = (uint32_t)f32_to_bf16(bacc[p][qt][2]) | ((uint32_t)f32_to_bf16(bacc[p][qt][3]) << 16);
      *reinterpret_cast<u32x2_t*>(&sh.u.bd[16 * kQT * w + 16 * qt + (l & 15)][16 * p + 4 * (l >> 4)]) = pk;
    }
  // a wave reads back only the rows it wrote (its LDS operations complete in order)
  // position term, mask, softmax (FP32), per query row
#pragma unroll
  for (int qt = 0; qt < kQT; ++qt) {
    const int i = 16 * kQT * w + 16 * qt + (l & 15);
    const uint16_t* bdr = &sh.u.bd[i][kAttT - 1 - i];
    float mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 8; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = 16 * kt + 4 * (l >> 4) + e;
        float s = acc[kt][qt][e] + bf16_to_f32(bdr[j]);
        if (j >= valid) s = -INFINITY;
        acc[kt][qt][e] = s;
        mx = fmaxf(mx, s);
      }
    mx = max_lanes16(mx);
    float z = 0.0f;
#pragma unroll
    for (int kt = 0; kt < 8; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p = expf(acc[kt][qt][e] - mx);
        acc[kt][qt][e] = p;
        z += p;
      }
    z = sum_lanes16(z);
#pragma unroll
    for (int kt = 0; kt < 8; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[kt][qt][e] = acc[kt][qt][e] / z;
  }
  // o^T = V^T . p^T: for key chunk c, a lane's eight k values are the keys
  // {16(2c) + 4(l/16) + e, 16(2c+1) + 4(l/16) + e} (e < 4) in both operands.
  f32x4_t o[kQT][8];
#pragma unroll
  for (int qt = 0; qt < kQT; ++qt)
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) o[qt][dt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int c = 0; c < kAttT / 32; ++c) {
    bf16x8_t phi[kQT], plo[kQT];
#pragma unroll
    for (int qt = 0; qt < kQT; ++qt) {
      uint32_t hw[4], lw[4];
#pragma unroll
      for (int e2 = 0; e2 < 4; ++e2) {
        uint16_t hi2[2], lo2[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int e = 2 * e2 + u;
          const float p = e < 4 ? acc[2 * c][qt][e] : acc[2 * c + 1][qt][e - 4];
          hi2[u] = f32_to_bf16(p);
          lo2[u] = f32_to_bf16(p - bf16_to_f32(hi2[u]));
        }
        hw[e2] = (uint32_t)hi2[0] | ((uint32_t)hi2[1] << 16);
        lw[e2] = (uint32_t)lo2[0] | ((uint32_t)lo2[1] << 16);
      }
      phi[qt] = as_bf16x8(uint4{hw[0], hw[1], hw[2], hw[3]});
      plo[qt] = as_bf16x8(uint4{lw[0], lw[1], lw[2], lw[3]});
    }
    const int j0 = 32 * c + 4 * (l >> 4);
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      const int d = 16 * dt + (l & 15);
      const uint32_t* vr = reinterpret_cast<const uint32_t*>(&sh.vt[d][0]);
      const bf16x8_t vf = as_bf16x8(uint4{vr[j0 / 2], vr[j0 / 2 + 1], vr[j0 / 2 + 8], vr[j0 / 2 + 9]});
#pragma unroll
      for (int qt = 0; qt < kQT; ++qt) {
        o[qt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, phi[qt], o[qt][dt], 0, 0, 0);
        o[qt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, plo[qt], o[qt][dt], 0, 0, 0);
      }
    }
  }
  // o[qt][dt]: lane l holds dimensions 16dt + 4(l/16) + e of query 16 kQT w + 16qt + l%16
#pragma unroll
  for (int qt = 0; qt < kQT; ++qt) {
    uint16_t* orow = out + (size_t)(b * kAttT + 16 * kQT * w + 16 * qt + (l & 15)) * kD + h * kDk + 4 * (l >> 4);
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      u32x2_t pk;
      pk.x = (uint32_t)f32_to_bf16(o[qt][dt][0]) | ((uint32_t)f32_to_bf16(o[qt][dt][1]) << 16);
      pk.y = (uint32_t)f32_to_bf16(o[qt][dt][2]) | ((uint32_t)f32_to_bf16(o[qt][dt][3]) << 16);
      *reinterpret_cast<u32x2_t*>(orow + 16 * dt) = pk;
    }
  }
}

// k_pk_attention_keys: a block takes 16 queries of one (sequence, head) and
// its four waves split the keys, 32 each, so one window runs on 64 CUs
// instead of 16. Bound by the latency of its one round of loads and of the
// two meetings of the waves. Nothing but the values is used twice by a wave,
// so keys, queries and the 48 rows of P_h^T that the shifted index
// T-1-i+j spans for them go from memory straight into MFMA operands, all of a
// block's loads in flight at once; the values are copied into the wave's LDS
// and read back transposed. The waves meet for the rows' maxima, and to add
// their partial values, which are divided by the rows' sums then. The
// exponentials carry a factor of 1 / 128 (exact), so that the undivided sums
// overflow no sooner than the values do.
constexpr int kAkWaves = 4, kAkQueries = 16;
constexpr int kAkThreads = kAkWaves * kWave;
constexpr int kAkKeys = kAttT / kAkWaves;    // keys per wave
constexpr int kAkBdRow = 48 + 4;             // bf16 per LDS row of a query's position scores
constexpr int kAkOutRow = kDk + 4;           // floats per LDS row of a query's partial values
struct PkAttKeysLds {
  union {
    uint4 v[kAkKeys * kDk / 8];              // the wave's values, then
    float out[kAkQueries][kAkOutRow];        // its partial results
  } w[kAkWaves];
  uint16_t bd[kAkWaves][kAkQueries][kAkBdRow];
  float top[kAkWaves][kAkQueries], sum[kAkWaves][kAkQueries];
};

// The transposing reads of 32 keys x 64 dimensions and the wait for them as
// one statement (as in the prompt pass's attention, lfm25_prompt.hip).
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void read_values(const uint32_t (&a)[4], s16x4 (&lo)[4], s16x4 (&hi)[4]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\t"
      "ds_read_b64_tr_b16 %1, %9\n\t"
      "ds_read_b64_tr_b16 %2, %10\n\t"
      "ds_read_b64_tr_b16 %3, %11\n\t"
      "ds_read_b64_tr_b16 %4, %8 offset:4096\n\t"
      "ds_read_b64_tr_b16 %5, %9 offset:4096\n\t"
      "ds_read_b64_tr_b16 %6, %10 offset:4096\n\t"
      "ds_read_b64_tr_b16 %7, %11 offset:4096\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(lo[0]), "=&v"(lo[1]), "=&v"(lo[2]), "=&v"(lo[3]), "=&v"(hi[0]), "=&v"(hi[1]), "=&v"(hi[2]), "=&v"(hi[3])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3])
      : "memory");
}

__global__ void __launch_bounds__(kAkThreads, 2)
    k_pk_attention_keys(const uint16_t* __restrict__ qkv, const uint16_t* __restrict__ pos,
                        const uint16_t* __restrict__ delta, uint16_t* __restrict__ out, int valid) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host pass has no LDS address space)
  __shared__ PkAttKeysLds sh;
  constexpr int kDs = kDk / 32;  // steps of 32 dimensions
  constexpr float kShare = 1.0f / kAttT;
  const int h = blockIdx.x, b = blockIdx.y, i0 = kAkQueries * blockIdx.z;
  const int t = threadIdx.x, w = wave_id(), l = lane_id(), col = l & 15, g = l >> 4;
  const uint16_t* base = qkv + (size_t)b * kAttT * 3 * kD + h * kDk;
  // values: key row r's chunk c in slot 16 r + (c ^ 2 (r % 8))
  {
    const uint16_t* v = base + 2 * kD + (size_t)kAkKeys * w * 3 * kD;
#pragma unroll
    for (int i = 0; i < kAkKeys * kDk / 8 / kWave; ++i) {
      const int slot = i * kWave + l, r = slot / 16, c = (slot % 16) ^ (2 * (r & 7));
      __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)(v + (size_t)r * 3 * kD + 8 * c),
                                       (tile::LdsVoid*)&sh.w[w].v[i * kWave], 16, 0, 0);
    }
  }
  uint4 q[kDs], k[2][kDs], p[3][kDs];
  const int p0 = kAttT - kAkQueries - i0 + kAkKeys * w;  // T-1-i+j of the last query and the wave's first key
#pragma unroll
  for (int ds = 0; ds < kDs; ++ds) {
    const int d = 32 * ds + 8 * g;
    q[ds] = *reinterpret_cast<const uint4*>(base + (size_t)(i0 + col) * 3 * kD + d);
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
      k[kt][ds] = *reinterpret_cast<const uint4*>(base + kD + (size_t)(kAkKeys * w + 16 * kt + col) * 3 * kD + d);
#pragma unroll
    for (int pt = 0; pt < 3; ++pt)
      p[pt][ds] = *reinterpret_cast<const uint4*>(pos + ((size_t)h * 2 * kAttT + p0 + 16 * pt + col) * kDk + d);
  }
  // position scores of query i0 + col and rows 16 pt + 4 g + e of the slice
#pragma unroll
  for (int pt = 0; pt < 3; ++pt) {
    f32x4_t a{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ds = 0; ds < kDs; ++ds)
      a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(p[pt][ds]), as_bf16x8(q[ds]), a, 0, 0, 0);
    *reinterpret_cast<uint2*>(&sh.bd[w][col][16 * pt + 4 * g]) =
        uint2{tile::pack_pair(a[0], a[1]), tile::pack_pair(a[2], a[3])};
  }
  // key scores: s[kt][e] of key 32 w + 16 kt + 4 g + e and query i0 + col
  f32x4_t s[2] = {f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}, f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
  for (int ds = 0; ds < kDs; ++ds) {
    const uint4 dl = *reinterpret_cast<const uint4*>(delta + h * kDk + 32 * ds + 8 * g);
    const uint32_t dw[4] = {dl.x, dl.y, dl.z, dl.w}, qw[4] = {q[ds].x, q[ds].y, q[ds].z, q[ds].w};
    uint32_t u[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = tile::pack_pair(lo_f32(qw[e]) + lo_f32(dw[e]), hi_f32(qw[e]) + hi_f32(dw[e]));
    const bf16x8_t qu = as_bf16x8(uint4{u[0], u[1], u[2], u[3]});
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
      s[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(k[kt][ds]), qu, s[kt], 0, 0, 0);
  }
  // position term and mask, then the rows' maxima over the waves
  float top = -INFINITY;
#pragma unroll
  for (int kt = 0; kt < 2; ++kt)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int j = 16 * kt + 4 * g + e;
      float v = s[kt][e] + bf16_to_f32(sh.bd[w][col][15 - col + j]);
      if (kAkKeys * w + j >= valid) v = -INFINITY;
      s[kt][e] = v;
      top = fmaxf(top, v);
    }
  top = max_lanes16(top);
  if (l < 16) sh.top[w][l] = top;
  lds_barrier();
#pragma unroll
  for (int u = 0; u < kAkWaves; ++u) top = fmaxf(top, sh.top[u][col]);
  float z = 0.0f;
  uint32_t hw[4], lw[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float e0 = kShare * expf(s[i / 2][2 * (i % 2)] - top), e1 = kShare * expf(s[i / 2][2 * (i % 2) + 1] - top);
    z += e0 + e1;
    hw[i] = tile::pack_pair(e0, e1);
    lw[i] = tile::pack_pair(e0 - lo_f32(hw[i]), e1 - hi_f32(hw[i]));
  }
  z = sum_lanes16(z);
  if (l < 16) sh.sum[w][l] = z;
  const bf16x8_t hi = as_bf16x8(uint4{hw[0], hw[1], hw[2], hw[3]}), lo = as_bf16x8(uint4{lw[0], lw[1], lw[2], lw[3]});
  // o^T = V^T . e^T over the wave's keys: a lane's eight k values are the keys
  // {4 g + e, 16 + 4 g + e} in both operands
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the wave's own value copies
  f32x4_t o[kDk / 16];
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    uint32_t at[4];
    const int vr = 4 * g + col / 4;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
      at[dt] = (uint32_t)(uintptr_t)(tile::LdsVoid*)&sh.w[w].v[16 * vr + ((8 * half + 2 * dt + (l & 3) / 2) ^ (2 * (vr & 7)))] + 8 * (l & 1);
    s16x4 v0[4], v1[4];
    read_values(at, v0, v1);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(v0[dt], v1[dt], 0, 1, 2, 3, 4, 5, 6, 7));
      f32x4_t a{0.0f, 0.0f, 0.0f, 0.0f};
      a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, hi, a, 0, 0, 0);
      o[4 * half + dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, lo, a, 0, 0, 0);
    }
  }
  // (over the wave's own values, which it has read)
#pragma unroll
  for (int dt = 0; dt < kDk / 16; ++dt) *reinterpret_cast<f32x4_t*>(&sh.w[w].out[col][16 * dt + 4 * g]) = o[dt];
  lds_barrier();
  // the waves' partials in order, over the row's sum: eight dimensions per thread
  const int qi = t / 16, d0 = 8 * (t % 16);
  float total = sh.sum[0][qi], v[8];
#pragma unroll
  for (int u = 1; u < kAkWaves; ++u) total += sh.sum[u][qi];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    v[e] = sh.w[0].out[qi][d0 + e];
#pragma unroll
    for (int u = 1; u < kAkWaves; ++u) v[e] += sh.w[u].out[qi][d0 + e];
    v[e] /= total;
  }
  tile::store_bf16<8>(out + (size_t)(b * kAttT + i0 + qi) * kD + h * kDk + d0, v, false);
#endif
}

// Blocks of 16 queries while they fit the chip twice (two of them to a CU):
// 6.4 us against 10.5 at one window, 6.7 / 10.7 at four, 9.9 / 11.4 at eight;
// at ten windows their third round makes it 12.7 against 11.1, at sixteen
// 16.0 against 11.8.
void launch_attention(const uint16_t* qkv, const uint16_t* pos, const uint16_t* delta, uint16_t* out, int batch,
                      int valid, hipStream_t s) {
  constexpr int kKeysBlocks = kPkHeads * (kAttT / kAkQueries);
  if (batch <= 2 * tile::kCus / kKeysBlocks)
    k_pk_attention_keys<<<dim3(kPkHeads, batch, kAttT / kAkQueries), kAkThreads, 0, s>>>(qkv, pos, delta, out, valid);
  else
    k_pk_attention<<<dim3(kPkHeads, batch, kAttSplit), kAttBlockThreads, 0, s>>>(qkv, pos, delta, out, valid);
}

// ------------------------------------------------------------------ conv module

// GLU + depthwise conv of 64 channels (blockIdx.x) over 32 frames
// (blockIdx.y) of sequence b (blockIdx.z), as the mirror
// (012_layer_test.py:92-100):
//   g_t = bf16(c_t[ch] * sigmoid(c_t[1024 + ch])) for t < valid, else 0;
//   y_t = sum_{j<9} g_{t+j-4} * dw[ch][j] (in order, zero outside the
//   frames) + bias[ch]; out = bf16(y * sigmoid(y)).
// Eight threads side by side take 64 adjacent channels of a frame, so every
// load and store covers whole 128-byte lines (with 16 channels a block they
// were 32-byte pieces of a 4 KB row, which bound the pass: 12.2 us at 16
// windows); the four frames to either side are formed twice.
constexpr int kConvCh = 64;
constexpr int kConvFrames = 32;
constexpr int kConvThreads = 256;
static_assert(kConvThreads == kConvFrames * kConvCh / 8, "a frame's eight channels per thread");
__global__ void __launch_bounds__(kConvThreads) k_pk_conv(const uint16_t* __restrict__ c, const uint16_t* __restrict__ dw,
                                                          const uint16_t* __restrict__ dw_b,
                                                          uint16_t* __restrict__ out, int valid) {
  constexpr int kHalo = kConvTapsPk / 2, kRows = kConvFrames + 2 * kHalo;
  __shared__ float g[kRows][kConvCh + 4];
  const int ch0 = blockIdx.x * kConvCh, t0 = blockIdx.y * kConvFrames, b = blockIdx.z, t = threadIdx.x;
  // this thread's channels ch0 + 8q .. + 7 and frame t0 + r
  const int q = t % (kConvCh / 8), r = t / (kConvCh / 8);
  const int ch = ch0 + 8 * q;
  const uint4* taps = reinterpret_cast<const uint4*>(dw + (size_t)ch * kConvTapsPk);  // 72 values, 9 x 16 bytes
  uint4 tap[kConvTapsPk];
#pragma unroll
  for (int u = 0; u < kConvTapsPk; ++u) tap[u] = taps[u];
  const uint4 bv = *reinterpret_cast<const uint4*>(dw_b + ch);
  // the GLU of rows r and (the last 8) r + 32; row i is frame t0 + i - 4
  const auto glu = [&](int i) {
    const int tt = t0 + i - kHalo;
    float v[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (tt >= 0 && tt < valid) {
      const uint16_t* row = c + (size_t)(b * kAttT + tt) * 2 * kD + ch;
      const uint4 av = *reinterpret_cast<const uint4*>(row);
      const uint4 gv = *reinterpret_cast<const uint4*>(row + kD);
      const uint32_t aw[4] = {av.x, av.y, av.z, av.w}, gw[4] = {gv.x, gv.y, gv.z, gv.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[2 * e] = round_bf16(tile::over_one_plus_exp(lo_f32(aw[e]), lo_f32(gw[e])));
        v[2 * e + 1] = round_bf16(tile::over_one_plus_exp(hi_f32(aw[e]), hi_f32(gw[e])));
      }
    }
    float4* dst = reinterpret_cast<float4*>(&g[i][8 * q]);
    dst[0] = float4{v[0], v[1], v[2], v[3]};
    dst[1] = float4{v[4], v[5], v[6], v[7]};
  };
  glu(r);
  if (r < 2 * kHalo) glu(r + kConvFrames);
  float wt[8][kConvTapsPk], bias[8];
#pragma unroll
  for (int u = 0; u < kConvTapsPk; ++u) {
    const uint32_t vw[4] = {tap[u].x, tap[u].y, tap[u].z, tap[u].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i0 = 8 * u + 2 * e;
      wt[i0 / kConvTapsPk][i0 % kConvTapsPk] = lo_f32(vw[e]);
      wt[(i0 + 1) / kConvTapsPk][(i0 + 1) % kConvTapsPk] = hi_f32(vw[e]);
    }
  }
  const uint32_t bw[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    bias[2 * e] = lo_f32(bw[e]);
    bias[2 * e + 1] = hi_f32(bw[e]);
  }
  __syncthreads();
  float y[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) y[k] = g[r][8 * q + k] * wt[k][0];
#pragma unroll
  for (int j = 1; j < kConvTapsPk; ++j)
#pragma unroll
    for (int k = 0; k < 8; ++k) y[k] = y[k] + g[r + j][8 * q + k] * wt[k][j];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    y[k] = y[k] + bias[k];
    y[k] = tile::over_one_plus_exp(y[k], y[k]);
  }
  tile::store_bf16<8>(out + (size_t)(b * kAttT + t0 + r) * kD + ch, y, true);
}

// ------------------------------------------------------------------ host

// Number of K splits for an m x n x k product: doubled while the grid has
// fewer blocks than the chip has CUs even with the smallest tile, each split
// keeping >= kMinChunk of K. (128 x 1024 x 4096 alone: 11.1 us unsplit, 6.8 /
// 4.8 / 4.9 in 2 / 4 / 8 splits; with K = 1024 4.5, 3.6 and 3.3 in 1, 2 and
// 4, where the fourth partial costs the pass that sums them as much.)
int pick_splits(int m, int n, int k) {
  int splits = 1;
  while (tile::blocks_of<tile::S32x64>(m, n) * 2 * splits <= tile::kCus && k % (2 * splits * kBK) == 0 &&
         k / (2 * splits) >= kMinChunk)
    splits *= 2;
  return splits;
}

template <int EPI, bool kSplit, bool kFar, typename S>
void launch_tiles(PkGemm g, int splits, hipStream_t s) {
  g.tiles = tile::tiles_of<S>(g.M, g.N, (int64_t)g.M * g.kchunk * 2);
  const int blocks = ahead_blocks(g.ahead, g.tiles.blocks(), S::kThreads);
  k_pk_gemm<EPI, kSplit, kFar, S><<<dim3(blocks, splits), S::kThreads, sizeof(tile::Lds<S>), s>>>(g);
}
template <int EPI, bool kSplit>
void launch_gemm(const PkGemm& g, int splits, hipStream_t s) {
  tile::with_shape(g.M, g.N, splits, [&](auto shape) { launch_tiles<EPI, kSplit, false, decltype(shape)>(g, splits, s); });
}
// Rows farther apart than a tile's 32-bit offsets reach (256 rows of kFarRows
// elements: 2 GB). Two tile shapes are enough for these: 128 x 128 x 8,192 in
// 1 / 8 splits 26 / 13 us, as near rows (an output per thread took 704).
constexpr int kFarRows = 1 << 22;
template <int EPI, bool kSplit>
void launch_far(const PkGemm& g, int splits, hipStream_t s) {
  if (tile::blocks_of<tile::S32x64>(g.M, g.N) * splits <= tile::kCus)
    launch_tiles<EPI, kSplit, true, tile::S32x64>(g, splits, s);
  else
    launch_tiles<EPI, kSplit, true, tile::S128x128>(g, splits, s);
}

template <int EPI>
void launch_splitk(dim3 grid, const float* part, int splits, int m, int n, const uint16_t* bias, uint16_t* c, int ldc,
                   hipStream_t s) {
  switch (partial_group(splits)) {
    case 1: k_pk_splitk<EPI, 1><<<grid, 256, 0, s>>>(part, splits, m, n, bias, c, ldc); break;
    case 2: k_pk_splitk<EPI, 2><<<grid, 256, 0, s>>>(part, splits, m, n, bias, c, ldc); break;
    case 4: k_pk_splitk<EPI, 4><<<grid, 256, 0, s>>>(part, splits, m, n, bias, c, ldc); break;
    default: k_pk_splitk<EPI, 8><<<grid, 256, 0, s>>>(part, splits, m, n, bias, c, ldc); break;
  }
}

// C = epi(A . Bt^T + bias), or (splits > 1) as `splits` K ranges through
// `part` (splits x m x n floats) and k_pk_splitk.
int gemm(const uint16_t* a, int lda, const uint16_t* bt, int ldb, const uint16_t* bias, uint16_t* c, int ldc, int m,
         int n, int k, int epi, int splits, float* part, hipStream_t s, const AheadPair& ahead = {}) {
  const bool wide = aligned16(c) && ldc % 8 == 0;
  const PkGemm g{a, bt, bias, c, part, 0.0f, lda, ldb, ldc, m, n, k / splits, wide, {}, splits > 1 ? AheadPair{} : ahead};
  const bool far = lda > kFarRows || ldb > kFarRows;
  if (splits > 1) {
    if (far) launch_far<EPI_NONE, true>(g, splits, s);
    else launch_gemm<EPI_NONE, true>(g, splits, s);
    const dim3 blocks((unsigned)m, (unsigned)((n / 4 + 255) / 256));
    switch (epi) {
      case EPI_NONE: launch_splitk<EPI_NONE>(blocks, part, splits, m, n, bias, c, ldc, s); break;
      case EPI_BIAS: launch_splitk<EPI_BIAS>(blocks, part, splits, m, n, bias, c, ldc, s); break;
      default: launch_splitk<EPI_SWISH>(blocks, part, splits, m, n, bias, c, ldc, s); break;
    }
  } else if (far) {
    switch (epi) {
      case EPI_NONE: launch_far<EPI_NONE, false>(g, 1, s); break;
      case EPI_BIAS: launch_far<EPI_BIAS, false>(g, 1, s); break;
      default: launch_far<EPI_SWISH, false>(g, 1, s); break;
    }
  } else {
    switch (epi) {
      case EPI_NONE: launch_gemm<EPI_NONE, false>(g, 1, s); break;
      case EPI_BIAS: launch_gemm<EPI_BIAS, false>(g, 1, s); break;
      default: launch_gemm<EPI_SWISH, false>(g, 1, s); break;
    }
  }
  return check_launch("parakeet gemm");
}

// One encoder product wider than d. Never split: at one window its smallest
// tiles already fill half the chip, and the pass that sums the partials
// would cost more than the other half gives.
// The weights of the two products after it are read ahead behind it.
struct EncWeights {
  const uint16_t* w;
  int n, k, splits;  // the product's n and k, and its K splits
};
EncWeights enc_ln_weights(const uint16_t* w, int rows, int k) { return {w, kD, k, pick_splits(rows, kD, k)}; }
int enc_gemm(const uint16_t* a, int lda, const uint16_t* bt, const uint16_t* bias, uint16_t* c, int ldc, int m, int n,
             int k, int epi, hipStream_t s, const EncWeights& next, const EncWeights& then) {
  AheadPair p{};
  const EncWeights* e[2] = {&next, &then};
  for (int i = 0; i < 2; ++i) {
    const int group = e[i]->w ? tile::ahead_group(m, e[i]->n, e[i]->splits, (int64_t)m * (e[i]->k / e[i]->splits) * 2) : 0;
    p.a[i] = Ahead{e[i]->w, group > 0 ? e[i]->n : 0, e[i]->k / 64, group > 0 ? group : 1};
  }
  return gemm(a, lda, bt, k, bias, c, ldc, m, n, k, epi, 1, nullptr, s, p);
}

struct ReduceLnArgs {
  const float* part;
  int splits;
  uint16_t* x;
  float scale;
  const uint16_t *g1, *b1, *g2, *b2;
  int normed_x;
  uint16_t* a;
  int rows;
};
template <int G>
void launch_reduce_ln(const ReduceLnArgs& r, hipStream_t s) {
  k_pk_reduce_ln<G><<<r.rows, kWave, 0, s>>>(r.part, r.splits, r.x, r.scale, r.g1, r.b1, r.g2,
                                                                   r.b2, r.normed_x, r.a, r.rows);
}

// A d-wide encoder product (m x 1024) whose end is a residual + LayerNorm:
// unsplit, the product's own epilogue updates x and k_pk_ln norms its rows;
// split (few rows), the FP32 partials go to `part` and k_pk_reduce_ln
// finishes the row.
int enc_gemm_ln(const uint16_t* a, int lda, const uint16_t* bt, int m, int k, float* part, uint16_t* x, float scale,
                const uint16_t* ln1, const uint16_t* ln2, int normed_x, uint16_t* out_a, hipStream_t s) {
  const int splits = pick_splits(m, kD, k);
  const PkGemm g{a, bt, nullptr, x, part, scale, lda, k, kD, m, kD, k / splits, true, {}, {}};
  const uint16_t* b2 = ln2 ? ln2 + kD : nullptr;
  if (splits == 1) {
    launch_gemm<EPI_RESIDUAL, false>(g, 1, s);
    k_pk_ln<<<(m + kLnRows - 1) / kLnRows, kLnRows * kWave, 0, s>>>(x, nullptr, 0.0f, ln1, ln1 + kD, ln2, b2, normed_x,
                                                                    out_a, m);
    return check_launch("parakeet gemm + layer norm");
  }
  launch_gemm<EPI_NONE, true>(g, splits, s);
  const ReduceLnArgs r{part, splits, x, scale, ln1, ln1 + kD, ln2, b2, normed_x, out_a, m};
  // a wave per block: latency-bound, all of a row's partials in flight at once
  if (splits == 2) launch_reduce_ln<2>(r, s);
  else launch_reduce_ln<4>(r, s);
  return check_launch("parakeet gemm + layer norm");
}

// FP32 partial buffer of the encoder. Split products (pick_splits) have at
// most kCus blocks of the smallest tile, 2 MB; callers are asked for what
// they always were, 32 MB or a float per row and channel.
constexpr size_t kPartBytes = (size_t)32 << 20;
static_assert((size_t)tile::kCus * tile::S32x64::kTM * tile::S32x64::kTN * sizeof(float) <= kPartBytes, "partials fit");
inline size_t pk_part_bytes(int rows) { return std::max(kPartBytes, (size_t)rows * kD * sizeof(float)); }

// Workspace of the encoder for `rows` = batch * 128 frames (bytes).
inline size_t pk_ws_bytes(int rows) {
  return pk_part_bytes(rows) + (size_t)rows * 2 * (kD /*a*/ + kPkFfn /*big*/ + kD /*o*/);
}

}  // namespace
}  // namespace lfm25

using namespace lfm25;

extern "C" {

int lfm25_pk_gemm(const uint16_t* a, int32_t lda, const uint16_t* bt, int32_t ldb, const uint16_t* bias, uint16_t* c,
                  int32_t ldc, int32_t m, int32_t n, int32_t k, int32_t epi, int32_t splits, void* workspace,
                  lfm25_stream_t stream) {
  LFM25_REQUIRE(a && bt && c, "pk gemm: null pointer");
  LFM25_REQUIRE(m >= 1 && n >= kBN && n % kBN == 0 && k >= kBK && k % kBK == 0,
                "pk gemm: need m >= 1, n a multiple of %d, k a multiple of %d (got %d, %d, %d)", kBN, kBK, m, n, k);
  LFM25_REQUIRE(lda >= k && ldb >= k && ldc >= n && lda % 8 == 0 && ldb % 8 == 0 && ldc % 4 == 0,
                "pk gemm: leading dimensions too small or misaligned");
  LFM25_REQUIRE(aligned16(a) && aligned16(bt) && (reinterpret_cast<uintptr_t>(c) & 7) == 0,
                "pk gemm: a, bt must be 16-byte and c 8-byte aligned");
  LFM25_REQUIRE(epi >= EPI_NONE && epi <= EPI_SWISH, "pk gemm: epilogue must be 0 (none), 1 (bias) or 2 (swish)");
  LFM25_REQUIRE(epi != EPI_BIAS || bias != nullptr, "pk gemm: bias epilogue needs a bias");
  LFM25_REQUIRE(splits >= 1 && k % (splits * kBK) == 0,
                "pk gemm: splits must divide k into multiples of %d (got %d splits of %d)", kBK, splits, k);
  LFM25_REQUIRE(splits == 1 || (workspace && aligned16(workspace)),
                "pk gemm: a split product needs a 16-byte aligned workspace of splits * m * n floats");
  return gemm(a, lda, bt, ldb, bias, c, ldc, m, n, k, epi, splits, static_cast<float*>(workspace),
              reinterpret_cast<hipStream_t>(stream));
}

int lfm25_pk_layer_norm(uint16_t* x, const uint16_t* y, float scale, const uint16_t* gamma1, const uint16_t* beta1,
                        const uint16_t* gamma2, const uint16_t* beta2, int32_t normed_x, uint16_t* a, int32_t rows,
                        lfm25_stream_t stream) {
  LFM25_REQUIRE(x && gamma1 && beta1 && rows >= 1, "pk layer norm: null pointer or no rows");
  LFM25_REQUIRE(normed_x || a != nullptr, "pk layer norm: the carry mode writes a");
  LFM25_REQUIRE(!gamma2 || (beta2 && a && normed_x), "pk layer norm: a second norm needs normed_x, beta2 and a");
  LFM25_REQUIRE(aligned16(x) && (!y || aligned16(y)) && (!a || aligned16(a)) && aligned16(gamma1) &&
                    aligned16(beta1) && (!gamma2 || (aligned16(gamma2) && aligned16(beta2))),
                "pk layer norm: rows and norm parameters must be 16-byte aligned");
  k_pk_ln<<<(rows + kLnRows - 1) / kLnRows, kLnRows * kWave, 0, reinterpret_cast<hipStream_t>(stream)>>>(
      x, y, scale, gamma1, beta1, gamma2, beta2, normed_x, a, rows);
  return check_launch("parakeet layer norm");
}

int lfm25_pk_attention(const uint16_t* qkv, const uint16_t* pos, const uint16_t* delta, uint16_t* out, int32_t batch,
                       int32_t frames, int32_t valid, lfm25_stream_t stream) {
  LFM25_REQUIRE(qkv && pos && delta && out, "pk attention: null pointer");
  LFM25_REQUIRE(frames == kAttT, "pk attention: frames must be %d (one padded block), got %d", kAttT, frames);
  LFM25_REQUIRE(batch >= 1 && valid >= 1 && valid <= frames, "pk attention: need batch >= 1 and 1 <= valid <= frames");
  LFM25_REQUIRE(aligned16(qkv) && aligned16(pos) && aligned16(delta) && (reinterpret_cast<uintptr_t>(out) & 7) == 0,
                "pk attention: qkv, pos, delta must be 16-byte and out 8-byte aligned");
  launch_attention(qkv, pos, delta, out, batch, valid, reinterpret_cast<hipStream_t>(stream));
  return check_launch("parakeet attention");
}

int lfm25_pk_conv(const uint16_t* c, const uint16_t* dw, const uint16_t* dw_b, uint16_t* out, int32_t batch,
                  int32_t frames, int32_t valid, lfm25_stream_t stream) {
  LFM25_REQUIRE(c && dw && dw_b && out, "pk conv: null pointer");
  LFM25_REQUIRE(frames == kAttT, "pk conv: frames must be %d, got %d", kAttT, frames);
  LFM25_REQUIRE(batch >= 1 && valid >= 1 && valid <= frames, "pk conv: need batch >= 1 and 1 <= valid <= frames");
  LFM25_REQUIRE(aligned16(c) && aligned16(dw) && aligned16(dw_b) && aligned16(out), "pk conv: 16-byte alignment");
  k_pk_conv<<<dim3(kD / kConvCh, kAttT / kConvFrames, batch), kConvThreads, 0, reinterpret_cast<hipStream_t>(stream)>>>(c, dw, dw_b, out,
                                                                                                   valid);
  return check_launch("parakeet conv");
}

size_t lfm25_pk_workspace_bytes(int32_t batch, int32_t frames) {
  if (batch < 1 || frames != kAttT) return 0;
  return pk_ws_bytes(batch * frames);
}

int lfm25_pk_encoder(const lfm25_pk_layer* layers, int32_t n_layers, uint16_t* x, int32_t batch, int32_t frames,
                     int32_t valid, void* workspace, lfm25_stream_t stream) {
  LFM25_REQUIRE(layers && x && workspace && n_layers >= 1, "pk encoder: null argument");
  LFM25_REQUIRE(frames == kAttT && batch >= 1 && valid >= 1 && valid <= frames,
                "pk encoder: frames must be %d and 1 <= valid <= frames", kAttT);
  LFM25_REQUIRE(aligned16(x) && aligned16(workspace), "pk encoder: x and workspace must be 16-byte aligned");
  for (int i = 0; i < n_layers; ++i) {
    const lfm25_pk_layer& L = layers[i];
    LFM25_REQUIRE(L.ln && L.ff1_w1 && L.ff1_w2 && L.qkv && L.qkv_bias && L.att_delta && L.pos && L.out && L.pw1 &&
                      L.dw && L.dw_b && L.pw2 && L.ff2_w1 && L.ff2_w2,
                  "pk encoder: layer %d has a null tensor", i);
    LFM25_REQUIRE(aligned16(L.ln) && aligned16(L.ff1_w1) && aligned16(L.ff1_w2) && aligned16(L.qkv) &&
                      aligned16(L.att_delta) && aligned16(L.pos) && aligned16(L.out) && aligned16(L.pw1) &&
                      aligned16(L.dw) && aligned16(L.dw_b) && aligned16(L.pw2) && aligned16(L.ff2_w1) &&
                      aligned16(L.ff2_w2),
                  "pk encoder: layer %d tensors must be 16-byte aligned", i);
  }
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int rows = batch * frames;
  char* ws = static_cast<char*>(workspace);
  float* part = reinterpret_cast<float*>(ws);
  uint16_t* a = reinterpret_cast<uint16_t*>(ws + pk_part_bytes(rows));
  uint16_t* big = a + (size_t)rows * kD;
  uint16_t* o = big + (size_t)rows * kPkFfn;
  int rc = LFM25_OK;
  auto ln_of = [](const lfm25_pk_layer& L, int which) { return L.ln + (size_t)which * 2 * kD; };
#define PK_TRY(call)               \
  do {                             \
    rc = (call);                   \
    if (rc != LFM25_OK) return rc; \
  } while (0)
  // a = LN_ff1(x) of the first layer; later layers get it from the previous
  // layer's last norm (LN_out, then the next LN_ff1, on the same row pass)
  k_pk_ln<<<(rows + kLnRows - 1) / kLnRows, kLnRows * kWave, 0, s>>>(x, nullptr, 0.0f, ln_of(layers[0], 0),
                                                                      ln_of(layers[0], 0) + kD, nullptr, nullptr, 0, a,
                                                                      rows);
  for (int i = 0; i < n_layers; ++i) {
    const lfm25_pk_layer& L = layers[i];
    const uint16_t* next_ln = i + 1 < n_layers ? ln_of(layers[i + 1], 0) : nullptr;
    // Macaron FFN 1: x = bf16(x + FFN(a) / 2), a = LN_att(x)
    PK_TRY(enc_gemm(a, kD, L.ff1_w1, nullptr, big, kPkFfn, rows, kPkFfn, kD, EPI_SWISH, s,
                    enc_ln_weights(L.ff1_w2, rows, kPkFfn), {L.qkv, 3 * kD, kD, 1}));
    PK_TRY(enc_gemm_ln(big, kPkFfn, L.ff1_w2, rows, kPkFfn, part, x, 0.5f, ln_of(L, 1), nullptr, 0, a, s));
    // relative-position self-attention: x = bf16(x + out(att)), a = LN_conv(x)
    PK_TRY(enc_gemm(a, kD, L.qkv, L.qkv_bias, big, 3 * kD, rows, 3 * kD, kD, EPI_BIAS, s,
                    enc_ln_weights(L.out, rows, kD), {L.pw1, 2 * kD, kD, 1}));
    launch_attention(big, L.pos, L.att_delta, o, batch, valid, s);
    PK_TRY(enc_gemm_ln(o, kD, L.out, rows, kD, part, x, 1.0f, ln_of(L, 2), nullptr, 0, a, s));
    // conv module: x = bf16(x + pw2(conv(pw1(a)))), a = LN_ff2(x)
    PK_TRY(enc_gemm(a, kD, L.pw1, nullptr, big, 2 * kD, rows, 2 * kD, kD, EPI_NONE, s,
                    enc_ln_weights(L.pw2, rows, kD), {L.ff2_w1, kPkFfn, kD, 1}));
    k_pk_conv<<<dim3(kD / kConvCh, kAttT / kConvFrames, batch), kConvThreads, 0, s>>>(big, L.dw, L.dw_b, o, valid);
    PK_TRY(enc_gemm_ln(o, kD, L.pw2, rows, kD, part, x, 1.0f, ln_of(L, 3), nullptr, 0, a, s));
    // Macaron FFN 2 and the block's output norm: x = LN_out(bf16(x + FFN(a) / 2)),
    // a = LN_ff1 of the next layer (x)
    PK_TRY(enc_gemm(a, kD, L.ff2_w1, nullptr, big, kPkFfn, rows, kPkFfn, kD, EPI_SWISH, s,
                    enc_ln_weights(L.ff2_w2, rows, kPkFfn), {i + 1 < n_layers ? layers[i + 1].ff1_w1 : nullptr, kPkFfn, kD, 1}));
    PK_TRY(enc_gemm_ln(big, kPkFfn, L.ff2_w2, rows, kPkFfn, part, x, 0.5f, ln_of(L, 4), next_ln, 1, a, s));
  }
#undef PK_TRY
  return check_launch("parakeet encoder");
}

}  // extern "C"
