// Reading the next product's weights ahead, out of HBM.
//
// A product of few rows is bound by its weights' way from HBM: its blocks
// start with nothing and the first bytes take 2-3 us (128 x 4096 x 1024 takes
// 4.8 us with its weights cached and 7.4 with them in HBM), while HBM idles
// most of the time. So a product carries extra blocks that touch each
// 128-byte line of the weights that the products after it will read. (Extra
// blocks in the short passes between products, norms and gates, made those
// passes as much longer as the products got shorter.) Every XCD has an L2 of
// its own; a product's blocks go to the XCDs round robin, so rows are dealt
// to the XCDs in groups of one tile: an extra block on XCD x touches the rows
// that the product's blocks on XCD x will read. (Where a block does not land
// on XCD blockIdx % 8 nothing but the gain is lost.) Measured: a prompt pass
// of 250 rows 718 -> 644 us, of 64 rows 619 -> 523, of 4 rows 585 -> 486; one
// encoder window 173 -> 170. (How much of it L2 gives and how much the
// memory-side cache behind it is not known: counters of single kernels show
// the lines fetched anew past L2.)
#pragma once
#include "lfm25_device.h"

namespace lfm25 {

constexpr int kXcds = 8;

// `rows` weight rows of `lines` 128-byte lines; row r goes to XCD (r / group)
// % 8. rows is a multiple of 8 * group. No rows: nothing to read.
struct Ahead {
  const uint16_t* w;
  int rows, lines, group;
};

// Extra blocks of `threads` threads for `a`: about four lines per thread.
inline int ahead_blocks(const Ahead& a, int threads) {
  const int per_xcd = a.rows / kXcds * a.lines;
  return kXcds * ((per_xcd + 4 * threads - 1) / (4 * threads));
}

// Two products' weights behind the `own` blocks of a kernel.
struct AheadPair {
  Ahead a[2];
  int second;  // the second's first block
};
inline int ahead_blocks(AheadPair& p, int own, int threads) {  // returns the kernel's whole grid
  p.second = own + ahead_blocks(p.a[0], threads);
  return p.second + ahead_blocks(p.a[1], threads);
}

// Block `first` + i of the kernel is extra block i of `blocks` (a multiple of 8).
__device__ __forceinline__ void read_ahead(const Ahead& a, int first, int blocks) {
  const int x = blockIdx.x % kXcds;
  const int at = ((int)blockIdx.x - first) / kXcds * blockDim.x + threadIdx.x, step = blocks / kXcds * blockDim.x;
  const int total = a.rows / kXcds * a.lines;
  uint32_t v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int l = min(at + i * step, total - 1), q = l / a.lines;
    const int row = (q / a.group * kXcds + x) * a.group + q % a.group;
    v[i] = *reinterpret_cast<const uint32_t*>(a.w + ((size_t)row * a.lines + l % a.lines) * 64);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) asm volatile("" ::"v"(v[i]));
}

// For the blocks past `own`.
__device__ __forceinline__ void read_ahead(const AheadPair& p, int own) {
  if ((int)blockIdx.x < p.second) read_ahead(p.a[0], own, p.second - own);
  else read_ahead(p.a[1], p.second, gridDim.x - p.second);
}

}  // namespace lfm25
