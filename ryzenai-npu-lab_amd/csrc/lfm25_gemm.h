// Matrix-core tile product shared by the Parakeet encoder and the prompt
// pass: C[m][n] = sum_k A[m][k] B[n][k] (BF16 operands, both contiguous along
// k, FP32 sums), one block tile of TM x TN per block.
//
// A block's waves form a kWM x kWN grid; a wave owns kMT x kNT MFMA tiles
// (v_mfma_f32_16x16x32_bf16, the B tile as the first operand). The operands
// are copied from global memory straight into LDS (buffer loads to LDS, 16
// bytes per lane) in kStages stages of one K step of 64.
//
// What bounds it, and why the loop looks as it does: at one wave per SIMD
// nothing else hides a wait, and the first form of this loop (read the
// fragments of a half step, wait, multiply) spent two thirds of its time in
// four exposed LDS round trips per step. Here every half step's 16-byte LDS
// reads are issued among the products of the half step before: the second
// half's fragments during the first half's products, and, past the one
// barrier in the middle of the step, the next step's first fragments during
// the second half's. At that barrier every wave holds all of the step's
// fragments in registers, so its LDS stage is free and the copies of step s +
// kStages go out right there; a copy has kStages - 1 steps to land.
#pragma once
#include "lfm25_device.h"

namespace lfm25 {
namespace tile {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef __attribute__((address_space(3))) void LdsVoid;

constexpr int kStep = 64;  // K elements per step: a tile row of eight 16-byte chunks
constexpr int kChunks = kStep / 8;

__device__ __forceinline__ Rsrc make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

template <int WM, int WN, int MT, int NT, int STAGES>
struct Shape {
  static constexpr int kWM = WM, kWN = WN, kMT = MT, kNT = NT, kStages = STAGES;
  static constexpr int kWaves = WM * WN, kThreads = kWaves * kWave;
  static constexpr int kTM = 16 * MT * WM, kTN = 16 * NT * WN;
  // copy instructions (64 chunks = 8 tile rows each) per wave and step
  static constexpr int kAI = kTM / 8 / kWaves, kBI = kTN / 8 / kWaves;
  static constexpr int kLaneN = 4 * NT;  // consecutive n that a lane's results of one row cover
  static_assert(kAI * 8 * kWaves == kTM && kBI * 8 * kWaves == kTN, "whole copy instructions per wave");
  static_assert(kWaves * (MT + NT) > 0 && STAGES >= 2, "stages");
};

// (In dynamic LDS: a static array past half of a CU's LDS makes the compiler
// plan for one wave per SIMD and 512 registers, and then move the results
// between the two halves of the register file every step.)
template <typename S>
struct Lds {
  uint4 a[S::kStages][S::kTM * kChunks];
  uint4 b[S::kStages][S::kTN * kChunks];
};

// Where chunk c of tile row r lies within the row's eight 16-byte slots: the
// 16 rows that an operand read touches at one chunk must differ in (row
// parity, slot), so that they spread over all 64 banks. An A tile's operand
// rows are consecutive. A B tile's are not: row 4g + b of MFMA tile t is tile
// row 4 kNT g + 4t + b, which gives a lane 4 kNT consecutive n of one m.
__device__ __forceinline__ int a_swizzle(int r) { return (r >> 1) & 7; }
template <typename S>
__device__ __forceinline__ int b_swizzle(int r) {
  return ((r >> 1) & 1) | (((r / S::kLaneN) & 3) << 1);
}

// Byte offsets of this lane's copies within the block's A and B tiles. A
// wave's copy instruction i fills slots (kAI w + i) * 64 + lane.
template <typename S>
struct Copies {
  int a[S::kAI], b[S::kBI];
};
// b_row(r) = the row, counted from the base of B's descriptor, of tile row r.
template <typename S, typename BRow>
__device__ __forceinline__ void copy_offsets(Copies<S>& c, int lda, int ldb, const BRow& b_row) {
  const int w = wave_id(), l = lane_id();
#pragma unroll
  for (int i = 0; i < S::kAI; ++i) {
    const int p = (S::kAI * w + i) * kWave + l, r = p / kChunks, q = (p % kChunks) ^ a_swizzle(r);
    c.a[i] = (r * lda + 8 * q) * 2;
  }
#pragma unroll
  for (int i = 0; i < S::kBI; ++i) {
    const int p = (S::kBI * w + i) * kWave + l, r = p / kChunks, q = (p % kChunks) ^ b_swizzle<S>(r);
    c.b[i] = (b_row(r) * ldb + 8 * q) * 2;
  }
}

// The same as 64-bit addresses, where rows lie farther apart than 32-bit
// offsets reach. Rows past `rows` repeat the last one.
template <typename S>
struct FarRows {
  const uint16_t *a[S::kAI], *b[S::kBI];
  __device__ __forceinline__ FarRows(const uint16_t* a_base, size_t lda, int rows, const uint16_t* b_base, size_t ldb) {
    const int w = wave_id(), l = lane_id();
#pragma unroll
    for (int i = 0; i < S::kAI; ++i) {
      const int p = (S::kAI * w + i) * kWave + l, r = p / kChunks, q = (p % kChunks) ^ a_swizzle(r);
      a[i] = a_base + min(r, rows - 1) * lda + 8 * q;
    }
#pragma unroll
    for (int i = 0; i < S::kBI; ++i) {
      const int p = (S::kBI * w + i) * kWave + l, r = p / kChunks, q = (p % kChunks) ^ b_swizzle<S>(r);
      b[i] = b_base + r * ldb + 8 * q;
    }
  }
};

// A wave's results: v[nt][mt][e] is C at row m = 16 (kMT wm + mt) + l % 16 and
// column n = 16 kNT wn + kLaneN (l / 16) + 4 nt + e of the block tile.
template <typename S>
struct Acc {
  f32x4 v[S::kNT][S::kMT];
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < S::kNT; ++i)
#pragma unroll
      for (int j = 0; j < S::kMT; ++j) v[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
};

// Spreads a half step's LDS reads, and then its kCopies copies, evenly over its
// products (the compiler keeps the copies behind the reads: both touch LDS).
template <typename S, int kCopies>
__device__ __forceinline__ void interleave() {
  constexpr int kReads = S::kMT + S::kNT, kMfma = S::kMT * S::kNT;
  constexpr int kShare = kCopies > 0 ? kMfma / 2 : kMfma;  // products that go with the reads
  constexpr int kGroups = kShare / 2 < kReads ? (kShare / 2 > 0 ? kShare / 2 : 1) : kReads;
#pragma unroll
  for (int i = 0; i < kGroups; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x100, (kReads + kGroups - 1) / kGroups, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, kShare / kGroups, 0);
  }
  if constexpr (kCopies > 0) {
    constexpr int kLeft = kMfma - kShare, kPairs = kLeft < kCopies ? kLeft : kCopies;
#pragma unroll
    for (int i = 0; i < kPairs; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x020, (kCopies + kPairs - 1) / kPairs, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, kLeft / kPairs, 0);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
}

// acc += the block tile's product over `steps` K steps. The
// descriptors cover the tile's rows inside the matrix (a lane offset past
// them touches no memory, and what its row's products are is not used; the
// step's offset is scalar and not checked). Or (kFar) all of it from `far`.
// Leaves no copy in flight.
template <typename S, bool kFar = false>
__device__ __forceinline__ void product(Lds<S>& sh, const void* a_base, uint32_t a_bytes, const void* b_base,
                                        uint32_t b_bytes, const Copies<S>& c, int steps, Acc<S>& acc,
                                        const FarRows<S>* far = nullptr) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host pass has no LDS address space)
  const int w = wave_id(), l = lane_id();
  const int wm = w % S::kWM, wn = w / S::kWM;
  // steps past the last copy nothing: an empty descriptor, so that every
  // step leaves the same number of loads to count (far rows: the last step
  // again, into a stage that nothing reads)
  const auto copy = [&](int step, int stage) {
    if constexpr (kFar) {
      typedef __attribute__((address_space(1))) void GlobalVoid;
      const int k = min(step, steps - 1) * kStep;
#pragma unroll
      for (int i = 0; i < S::kAI; ++i)
        __builtin_amdgcn_global_load_lds((GlobalVoid*)(far->a[i] + k), (LdsVoid*)&sh.a[stage][(S::kAI * w + i) * kWave], 16, 0, 0);
#pragma unroll
      for (int i = 0; i < S::kBI; ++i)
        __builtin_amdgcn_global_load_lds((GlobalVoid*)(far->b[i] + k), (LdsVoid*)&sh.b[stage][(S::kBI * w + i) * kWave], 16, 0, 0);
      return;
    }
    const bool in = step < steps;
    const Rsrc ra = make_rsrc(a_base, in ? a_bytes : 0), rb = make_rsrc(b_base, in ? b_bytes : 0);
    const int k = in ? step * kStep * 2 : 0;
#pragma unroll
    for (int i = 0; i < S::kAI; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (LdsVoid*)&sh.a[stage][(S::kAI * w + i) * kWave], 16, c.a[i], k, 0, 0);
#pragma unroll
    for (int i = 0; i < S::kBI; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (LdsVoid*)&sh.b[stage][(S::kBI * w + i) * kWave], 16, c.b[i], k, 0, 0);
  };
  // slot of this lane's operand rows at chunk l / 16 (+ 4 for the second half)
  int ar[2], br[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int kc = 4 * h + (l >> 4);
    const int ra = 16 * S::kMT * wm + (l & 15);
    ar[h] = ra * kChunks + (kc ^ a_swizzle(ra));
    const int rb = 16 * S::kNT * wn + S::kLaneN * ((l & 15) >> 2) + (l & 3);
    br[h] = rb * kChunks + (kc ^ b_swizzle<S>(rb));
  }
  const auto fragments = [&](int stage, int h, bf16x8 (&xa)[S::kMT], bf16x8 (&wb)[S::kNT]) {
    // rows 16 apart keep a_swizzle, rows 4 apart within a lane's run keep b_swizzle
#pragma unroll
    for (int i = 0; i < S::kMT; ++i) xa[i] = __builtin_bit_cast(bf16x8, sh.a[stage][ar[h] + 16 * i * kChunks]);
#pragma unroll
    for (int i = 0; i < S::kNT; ++i) wb[i] = __builtin_bit_cast(bf16x8, sh.b[stage][br[h] + 4 * i * kChunks]);
  };
  const auto multiply = [&](const bf16x8 (&xa)[S::kMT], const bf16x8 (&wb)[S::kNT]) {
#pragma unroll
    for (int nt = 0; nt < S::kNT; ++nt)
#pragma unroll
      for (int mt = 0; mt < S::kMT; ++mt)
        acc.v[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[nt], xa[mt], acc.v[nt][mt], 0, 0, 0);
  };
  constexpr int kPer = S::kAI + S::kBI;  // copies per step and wave
#pragma unroll
  for (int i = 0; i < S::kStages; ++i) copy(i, i);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kPer * (S::kStages - 1)) : "memory");
  bf16x8 xa0[S::kMT], wb0[S::kNT], xa1[S::kMT], wb1[S::kNT];
  fragments(0, 0, xa0, wb0);
  int stage = 0;
  for (int s = 0; s < steps; ++s) {
    const int next = stage + 1 == S::kStages ? 0 : stage + 1;
    fragments(stage, 1, xa1, wb1);
    multiply(xa0, wb0);
    interleave<S, 0>();
    // This wave's copies of step s + 1 have landed (those of later steps may
    // be in flight) and its reads of step s are in registers; behind the
    // barrier every wave's are.
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kPer * (S::kStages - 2)) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    fragments(next, 0, xa0, wb0);  // (past the last step: read, never used)
    copy(s + S::kStages, stage);
    multiply(xa1, wb1);
    interleave<S, kPer>();
    stage = next;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the last copies' LDS writes, before the block's LDS is given back
#endif
}

// f(m, n, v) for each row m < rows of the wave's results: v[0 .. kLaneN) are
// the columns n .. n + kLaneN - 1 of the block tile at (m0, n0).
template <typename S, typename F>
__device__ __forceinline__ void each_row(const Acc<S>& acc, int m0, int n0, int rows, const F& f) {
  const int w = wave_id(), l = lane_id();
  const int wm = w % S::kWM, wn = w / S::kWM;
  const int n = n0 + 16 * S::kNT * wn + S::kLaneN * (l >> 4);
#pragma unroll
  for (int mt = 0; mt < S::kMT; ++mt) {
    const int m = m0 + 16 * (S::kMT * wm + mt) + (l & 15);
    if (m >= rows) continue;
    float v[S::kLaneN];
#pragma unroll
    for (int nt = 0; nt < S::kNT; ++nt)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * nt + e] = acc.v[nt][mt][e];
    f(m, n, v);
  }
}

// Two floats as a BF16 pair, low first: one v_cvt_pk_bf16_f32 (two separate
// conversions become two of them and two more to join the halves).
__device__ __forceinline__ uint32_t pack_pair(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}

// kN consecutive values as BF16 pairs; p is 8-byte aligned, 16-byte where
// `wide` (16-byte stores need it).
template <int kN>
__device__ __forceinline__ void store_bf16(uint16_t* p, const float (&v)[kN], bool wide) {
  uint32_t o[kN / 2];
#pragma unroll
  for (int i = 0; i < kN / 2; ++i) o[i] = pack_pair(v[2 * i], v[2 * i + 1]);
  if constexpr (kN % 8 == 0) {
    if (wide) {
#pragma unroll
      for (int i = 0; i < kN / 8; ++i)
        reinterpret_cast<uint4*>(p)[i] = uint4{o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]};
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < kN / 4; ++i) reinterpret_cast<uint2*>(p)[i] = uint2{o[2 * i], o[2 * i + 1]};
}
// kN consecutive BF16 values, p aligned as for store_bf16's wide form.
template <int kN>
__device__ __forceinline__ void load_bf16(const uint16_t* p, float (&v)[kN]) {
  if constexpr (kN % 8 == 0) {
#pragma unroll
    for (int i = 0; i < kN / 8; ++i) unpack8(load8(p + 8 * i), v + 8 * i);
  } else {
    const uint2 r = *reinterpret_cast<const uint2*>(p);
    v[0] = lo_f32(r.x); v[1] = hi_f32(r.x); v[2] = lo_f32(r.y); v[3] = hi_f32(r.y);
  }
}

// v / (1 + e^-x): sigmoid gates, and Swish / SiLU with v = x. expf and an
// IEEE division are about 30 instructions a value (6 us of a 2048 x 4096
// product's 29); this is 12. e^-x is 2^t, t = -x log2(e) rounded, times 1 +
// ln(2) times what t's rounding left out; 1 + e^-x is held scaled by 2^-24,
// so that e^-x does not overflow, nor its reciprocal become a denormal number
// that v_rcp flushes, where the result is still a normal one. t is rounded
// to 2^-14 (the FP32 step at kGrid), so that t - 24 is exact (rounding t and
// then t - 24 costs up to 14 x 2^-24). Within 7 x 2^-24 of the exact value (a
// unit in the last place of the exponential and of the reciprocal, three
// roundings); over 3.6 million numbers from -16 to 16 29 BF16 results are not
// the nearest, as in the expf form (96 with t and t - 24 both rounded).
// Infinities and NaN give what the expf form gave: x itself goes into the
// exponent, and only what t left out is clamped (it is below 2^-13 where the
// result is neither 0 nor v, and a NaN at an infinite x).
__device__ __forceinline__ float over_one_plus_exp(float v, float x) {
  constexpr float kLog2e = 0x1.715476p+0f, kLog2eRest = 0x1.4ae0cp-26f, kLn2 = 0x1.62e43p-1f, kScale = 0x1p-24f;
  constexpr float kGrid = 768.0f;
  const float t24 = fmaf(-x, kLog2e, kGrid - 24.0f) - kGrid;  // t - 24
  const float rest = __builtin_amdgcn_fmed3f(fmaf(-x, kLog2eRest, fmaf(-x, kLog2e, -24.0f - t24)), -1.0f, 1.0f);
  const float d = fmaf(__builtin_amdgcn_exp2f(t24), fmaf(rest, kLn2, 1.0f), kScale);
  return v * (__builtin_amdgcn_rcpf(d) * kScale);
}

// The tile shapes and the rule that picks one for an m x n product of
// `splits` K ranges: the smallest tile whose blocks number at most one per
// CU, so that a small product spreads over the chip and a large one reads
// fewer bytes per product; past that the largest tile where it fills whole
// rounds of the chip, else two resident 128 x 128 blocks, one multiplying
// while the other waits or stores. Measured alone, back to back, the weights
// from HBM (us; the column that the rule takes marked *):
//   m x n x k             32x64   64x64  64x128  128x128  256x128  128x128 twice
//   128 x 1024 x 1024      4.5*    5.4     6.4      8.7
//   128 x 4096 x 1024      4.8*    5.6     6.6      8.9
//   250 x 5120 x 1024      8.6     7.5     7.1*     9.3               9.9
//   640 x 3072 x 1024     11.5     8.1     7.7*     9.8
//   640 x 5120 x 1024     18.4    14.3    11.6     10.4*
//   2048 x 1024 x 4096                    25.9*    34.8     48.2     57.4
//   2048 x 2048 x 1024                    16.1     12.6*    17.3     18.4
//   2048 x 3072 x 1024                    22.2     22.3     18.2*    20.7
//   2048 x 4096 x 1024                    29.5     25.4     19.6*    22.1
//   3900 x 5120 x 1024                    64.7     49.4     47.0*    48.6
// (torch.matmul, that is hipBLASLt, on 2048 x 4096 x 1024: 21.6.)
typedef Shape<1, 4, 2, 1, 4> S32x64;
typedef Shape<2, 2, 2, 2, 4> S64x64;
typedef Shape<2, 4, 2, 2, 5> S64x128;
typedef Shape<2, 4, 4, 2, 3> S128x128;
typedef Shape<2, 4, 4, 2, 2> S128x128Twice;
typedef Shape<4, 2, 4, 4, 3> S256x128;
constexpr int kCus = 256;

template <typename S>
inline int64_t blocks_of(int m, int n) { return (int64_t)((m + S::kTM - 1) / S::kTM) * (n / S::kTN); }

// Calls f(shape) with the shape for the product (n a multiple of 128).
template <typename F>
inline void with_shape(int m, int n, int splits, const F& f) {
  const int64_t largest = blocks_of<S256x128>(m, n) * splits, rounds = (largest + kCus - 1) / kCus;
  if (blocks_of<S32x64>(m, n) * splits <= kCus) f(S32x64{});
  else if (blocks_of<S64x64>(m, n) * splits <= kCus) f(S64x64{});
  else if (blocks_of<S64x128>(m, n) * splits <= kCus) f(S64x128{});
  else if (blocks_of<S128x128>(m, n) * splits <= kCus) f(S128x128{});
  else if (rounds == 1 || 5 * largest >= 4 * rounds * kCus) f(S256x128{});
  else f(S128x128Twice{});
}

// Which tile a block takes. Blocks go to the eight XCDs round robin, each
// with its own 4 MB L2. In the plain order (n tiles fastest) an XCD reads all
// of A and an eighth of B; where A is larger than its L2, the tiles are dealt
// out as 2 x 4 rectangles, one per XCD, which reads half of A and a quarter
// of B: 2048 x 1024 x 4096 28.4 -> 25.9 us, 3900 x 1024 x 2560 28.1 -> 25.7
// (with A of 4 MB it gains nothing: 2048 x 4096 x 1024 19.6 -> 20.9).
struct Tiles {
  int m, n;     // tiles
  bool rects;
  __host__ __device__ int rect_m() const { return (m + 1) / 2; }
  __host__ __device__ int rect_n() const { return (n + 3) / 4; }
  __host__ __device__ int blocks() const { return rects ? 8 * rect_m() * rect_n() : m * n; }
  // False for a block past the tiles (a rectangle that sticks out).
  __device__ bool of(int block, int& tm, int& tn) const {
    if (!rects) {
      tn = block % n;
      tm = block / n;
      return true;
    }
    const int x = block % 8, i = block / 8;
    tm = (x / 4) * rect_m() + i / rect_n();
    tn = (x % 4) * rect_n() + i % rect_n();
    return tm < m && tn < n;
  }
};
template <typename S>
inline Tiles tiles_of(int m, int n, int64_t a_bytes) {
  const int tm = (m + S::kTM - 1) / S::kTM, tn = n / S::kTN;
  return Tiles{tm, tn, a_bytes > (4 << 20) && tm >= 8 && tn >= 4};
}

// The tile width of an m-row product whose weights' way from HBM bounds it
// (their rows go to the XCDs in groups of it), or 0: not where the products
// are long enough to hide it (1,024 rows and more), nor where the tiles are
// dealt out in another order.
inline int ahead_group(int m, int n, int splits, int64_t a_bytes) {
  if (m > 1024) return 0;
  int group = 0;
  with_shape(m, n, splits, [&](auto shape) {
    const Tiles t = tiles_of<decltype(shape)>(m, n, a_bytes);
    group = t.rects || t.n % 8 != 0 ? 0 : decltype(shape)::kTN;
  });
  return group;
}

}  // namespace tile
}  // namespace lfm25
