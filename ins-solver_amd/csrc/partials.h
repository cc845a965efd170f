// How many partial sums the kernels leave, and the room that a solver keeps for them. Host code alone:
// the counts are checked against the room for every order and mesh size on the CPU.
#pragma once

#include <algorithm>
#include <cstdint>

namespace insp {

constexpr int kRedBlocks = 8192;  // partials per reduction slot (vector kernels)
constexpr int kPartBlock = 256;   // threads of a block that leaves a partial

// Element passes: one thread per cell, or four waves per 64 cells.
inline int64_t one_thread_blocks(int64_t E) { return (E + kPartBlock - 1) / kPartBlock; }
inline int64_t four_wave_blocks(int64_t E) { return (E + 63) / 64; }

// Pairs of entries per thread of the coarse CG's streams, on n2 pairs: one, two or four while that leaves
// about a thousand blocks, whose partials (and their reading of others') are cheap; longer vectors
// stream at two per thread and leave the partials to a kernel in between. us per coarse iteration, 3D
// order 1: 547k cells with two per thread and finalize 57.3, four and folded 54.5; 1.57M cells 157.4,
// eight and folded 161.1.
inline int cg_pairs(int64_t n2) {
  if (n2 <= (int64_t)kPartBlock * 1024) return 1;
  if (n2 <= (int64_t)kPartBlock * 2 * 1024 || n2 > (int64_t)kPartBlock * 4 * 1536) return 2;
  return 4;
}
inline int64_t cg_blocks(int64_t n2, int per) { return (n2 + (int64_t)kPartBlock * per - 1) / ((int64_t)kPartBlock * per); }
// Blocks of those streams on vectors of n entries: one partial each, with no upper limit.
inline int64_t cg_stream_blocks(int64_t n) { return cg_blocks(n / 2, cg_pairs(n / 2)); }

// Whether every block of a consumer adds so many partials itself, rather than a kernel of its own in front of
// it: up to 35 MB of them read from L2 in all. us per two coarse iterations at 3D order 1, FP64, both sums
// by a kernel / folded: 235,824 cells 55.3 / 51.0, 663,552 (3.4 M partials read for p.Ap) 112.0 / 110.3,
// 750,000 (4.3 M) 123.5 / 119.0, 843,648 (10.9 M) 134 / 148; 2D 720,000 (3.0 M) 87.6 / 85.4.
constexpr int64_t kFoldReads = 4400000;
inline bool fold_pays(int64_t parts, int64_t blocks) { return parts * blocks <= kFoldReads; }
// The Jacobi and inverse-mass CG's three sums for the direction pass. us per iteration, kernel / folded: 3D
// order 2, 162,000 cells, inverse mass (6.0 M) 90.0 / 89.4; 3D order 4, 93,750 (7.1 M) 312.4 / 313.1; 3D order
// 3, 162,000 (12.0 M) 183.4 / 183.6; 3D order 4, 235,824 (45 M) 704 / 713; Jacobi, 2D order 4, 80,000 (8.3 M)
// 69.6 / 70.7.
constexpr int kFoldParts = 1024;  // p.Ap of those, for the step's blocks
constexpr int64_t kPcgFoldReads = 6500000;
inline bool pcg_fold_pays(int64_t parts, int64_t blocks) { return 3 * parts * blocks <= kPcgFoldReads; }

// Blocks of the Jacobi CG's stream of n2 pairs: at most 1024 while a thread has at most two pairs.
inline int64_t pcg_stream_blocks(int64_t n2) {
  const int64_t one = (n2 + kPartBlock - 1) / kPartBlock;
  if (one <= 2048) return std::max<int64_t>(1, std::min<int64_t>(one, 1024));
  return std::min<int64_t>((one + 1) / 2, kRedBlocks);
}

// Doubles in each half of a solver's partial sums (the coarse CG leaves two sums at a time, the Jacobi and
// inverse-mass CG the element pass's beside three of its own, the vector kernels four slots), on E
// cells and vectors of at most n entries. The coarse CG may run on any order: from order 3 on in 3D its
// streams leave more partials than the element passes do.
inline int64_t partials_half(int64_t E, int64_t n) {
  return std::max({(int64_t)4 * kRedBlocks, four_wave_blocks(E), cg_stream_blocks(n)});
}

}  // namespace insp
