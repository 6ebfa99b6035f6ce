// How a launch over token tiles deals its work out to the 8 XCDs. Plain integer arithmetic, for the host as well.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define BP_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define BP_HOST_DEVICE inline
#endif

namespace bp {

// Workgroups are dealt to the XCDs round-robin by linear index and each XCD has its own L2. A launch without a tile list has
// (expert, token tile, row block) triples: the row blocks of a tile read the same activations, the tiles of an expert the same
// weights. They are put in one sequence, of which XCD x takes the x-th contiguous eighth: a tile's row blocks are neighbours,
// then a run's tiles (64 token rows of an expert), and the runs are ordered so that an eighth is what one XCD should have:
//  * whole groups of eight experts: class c of the group i holds run 0 of expert 8 i + c, run 1 of expert 8 i + c - 1 (mod 8), ...
//    Neighbouring experts fall on different XCDs, and an expert with many rows is spread over them by runs, whichever
//    experts those are (a launch often has few experts with rows, next to each other or at some stride);
//  * the E % 8 experts that are left over, or a launch of fewer than eight (one: a dense linear): one after the other, in
//    whole, so that the eighths are equal whatever E is.
// 64 experts x 2048 x 2048, 4096 rows, us (whole experts dealt by expert % 8 / the triples in plain expert order / this order): TQ1, bf16:
// 64 rows each 108 / 111 / 103; 512 rows in eight neighbours 121 / 795 / 118, in every eighth expert 786 / 123 / 120; 1 to 127 rows,
// ascending, 143 / 182 / 136. TQ2, int8, 512 rows in eight neighbours 92 / 330 / 87. Runs of 128 rows: in every eighth expert 209, the
// rest level or 1 - 5 % slower.
//
// The divisions go by precomputed reciprocals: six divisions by variables ahead of a workgroup's first load took 2 - 4 % of a launch of a
// few rounds of workgroups (8 x 512 rows of the above, TQ2 with bf16 activations, 108.8 us against 102.5).
struct Divisor {  // n / d for n < 2^31: (n * m) >> (31 + s), 2^s >= d, m = 2^(31 + s) / d rounded up (its excess times n stays below 2^(31 + s))
  unsigned m, s;
};
inline Divisor divisor(unsigned d) {
  Divisor v = {0, 0};
  if (d == 0) return v;
  while ((1ull << v.s) < d) ++v.s;
  v.m = (unsigned)(((1ull << (31 + v.s)) + d - 1) / d);
  return v;
}
BP_HOST_DEVICE unsigned quotient(unsigned n, const Divisor& d) { return (unsigned)(((uint64_t)n * d.m) >> (31 + d.s)); }

struct TileSplit {
  unsigned experts, tiles_per_expert, tiles_per_run, runs;  // runs of an expert
  unsigned row_blocks, eighth;                              // items of an XCD
  Divisor by_blocks, by_tiles, by_runs, by_class, by_class1;  // (class: a group of eight's share, class1: with one of the experts left over)
};
inline TileSplit tile_split(int64_t E, int64_t max_rows, int tile_rows, int64_t row_blocks) {
  TileSplit s = {};
  s.experts = (unsigned)E;
  s.tiles_per_expert = (unsigned)((max_rows + tile_rows - 1) / tile_rows);
  const unsigned most = tile_rows >= 64 ? 1u : 64u / (unsigned)tile_rows;
  s.runs = E < 8 ? 1u : (s.tiles_per_expert + most - 1) / most;
  s.tiles_per_run = s.runs ? (s.tiles_per_expert + s.runs - 1) / s.runs : 0u;
  s.row_blocks = (unsigned)row_blocks;
  s.by_blocks = divisor(s.row_blocks);
  s.by_tiles = divisor(s.tiles_per_run);
  s.by_runs = divisor(s.runs);
  s.by_class = divisor((s.experts >> 3) * s.runs);
  s.by_class1 = divisor((s.experts >> 3) * s.runs + s.runs);
  return s;
}
// Items of the whole sequence, a multiple of 8 (-1: more than a grid's x extent holds). Some are empty (tile_item: false).
inline int64_t tile_items(const TileSplit& s) {
  const int64_t per_expert = (int64_t)s.runs * s.tiles_per_run, row_blocks = s.row_blocks;
  if (per_expert > 0x7ffffff8 / row_blocks || (int64_t)s.experts > 0x7ffffff8 / (row_blocks * (per_expert > 0 ? per_expert : 1))) return -1;
  return ((int64_t)s.experts * per_expert * row_blocks + 7) & ~(int64_t)7;
}
// The triple of workgroup `linear` (s.eighth: an eighth of the items); false: none.
BP_HOST_DEVICE bool tile_item(const TileSplit& s, unsigned linear, unsigned& expert, unsigned& tile, unsigned& row_block) {
  const unsigned item = (linear & 7) * s.eighth + (linear >> 3);
  const unsigned at = quotient(item, s.by_blocks);
  row_block = item - at * s.row_blocks;
  if (s.experts == 1) {  // (a dense call)
    expert = 0;
    tile = at;
    return tile < s.tiles_per_expert;
  }
  unsigned run = quotient(at, s.by_tiles);
  tile = at - run * s.tiles_per_run;
  const unsigned whole = s.experts >> 3, left = s.experts & 7;  // groups of eight, experts past them
  // the classes in order: the first `left` of them hold one of the experts that are left over as well
  const unsigned len = whole * s.runs, len1 = len + s.runs;
  unsigned c;
  if (run < left * len1) {
    c = quotient(run, s.by_class1);
    run -= c * len1;
  } else {
    if (len == 0) return false;
    run -= left * len1;
    const unsigned k = quotient(run, s.by_class);
    c = left + k;
    run -= k * len;
    if (c >= 8) return false;
  }
  if (run < len) {
    const unsigned i = quotient(run, s.by_runs), r = run - i * s.runs;
    expert = 8 * i + ((c - r) & 7);
    tile += r * s.tiles_per_run;
  } else {
    expert = 8 * whole + c;
    tile += (run - len) * s.tiles_per_run;
  }
  return tile < s.tiles_per_expert;
}

// With a list of the token tiles that exist, in expert order: an XCD takes the list in runs of 128 token rows, a tile's row
// blocks one after the other. (Runs of four tiles whatever their rows left a layer with 16 tiles of 128 to four XCDs: 8 experts
// top-2, 1024 rows, hidden 7168 / intermediate 2048, int8, 287 us against 177.)
BP_HOST_DEVICE unsigned list_item(const TileSplit& s, int tile_rows, unsigned linear, unsigned& row_block) {
  const unsigned run = 128u / (unsigned)tile_rows, xcd = linear & 7, q = linear >> 3, at = quotient(q, s.by_blocks);
  row_block = q - at * s.row_blocks;
  return at / run * (8 * run) + xcd * run + at % run;
}
// Workgroups for a list of up to `cap` tiles (-1: as above); positions past the list's end hold no tile.
inline int64_t list_items(int tile_rows, int64_t cap, int64_t row_blocks) {
  const int64_t per = 8 * (128 / tile_rows), rounds = (cap + per - 1) / per;
  return rounds > 0x7fffffff / (row_blocks * per) ? -1 : row_blocks * per * rounds;
}

}  // namespace bp
