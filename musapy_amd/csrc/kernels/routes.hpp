// routes.hpp -- which kernel variant a launch takes, from its plan alone (pure C++, like plan.hpp).
#pragma once

#include "plan.hpp"

namespace mpy {

inline uint64_t ceil_div(uint64_t a, uint64_t b) { return (a + b - 1) / b; }
inline uint32_t gcd32(uint32_t a, uint32_t b) { return b == 0 ? a : gcd32(b, a % b); }

// ---------------------------------------------------------------------------------------------
// How a column reduction (strided axis, unit-stride outputs) runs.  Three kernels share the shapes;
// the lines between them are those of a sweep over 1 to 20000 slices of 5 to 500000 rows of 8 to
// 600000 columns (f32 and f64, sums and max), and every figure below is from it.  `vecs` counts the
// 16-byte vectors of a row, `items` those of all slices.
//  * lanes: one lane per vector walks the whole axis.  It needs many of them (65536 lanes are one wave
//    per SIMD); then it is level with the column kernel or ahead of it, most where that one leaves lanes
//    idle or has less than a round of rows: (20000, 16, 8) sum 44.6 -> 7.3 us, (1000, 16, 512) max 13.2
//    -> 8.1.  With fewer the column kernel keeps more loads in flight ((256, 500, 512) max 44.8 against
//    73 us), and rows that fill its lanes only in part want 262144: (4000, 100, 300) sum 99 -> 82 us,
//    but (4000, 100, 100) 27 -> 32.
//  * spans: a block reads a whole number of rows per step.  They pay where the column kernel's 64 lanes
//    do not fill ((256, 4000, 8) sum 67.6 -> 9.1 us), or where one or a few slices leave it strips that
//    are far apart in memory ((30000, 512) sum 32 -> 14); with many slices of full rows they only cost
//    ((64, 100, 1000) sum 7.2 -> 14.6, (120, 2000, 1024) 145 -> 183).  Max / min / arg over one slice
//    keep the column kernel unless the array is long: (4000, 128) 9.0 us, 16.3 by spans.
//    25 to 63 blocks of the column kernel split into tiles that rarely come to one per CU: (18, 5000, 600)
//    f32 sum 59 us, 40 by spans, (10, 2100, 700) max 22.4 and 17.7, but (8, 5000, 1000), 256 blocks, 30 and 36.
//    Inputs of at most 4 MB split by column strips instead of row tiles, which saves the second
//    launch, if a strip is at most one and a half rounds long: (600, 400) sum 7.3 -> 5.4 us, but (3000,
//    100) 11.7 by columns, 13.7 by strips and 9.3 by tiles.
//  * columns: the 64-lane column kernel, for everything else.
struct ColRoute {
  enum : int { kColumns = 0, kLanes = 1, kSpans = 2 };
  int kind = kColumns;
  uint32_t bs = 0, cw = 0, strips = 1, m = 0, lanes = 0, tiles = 1;
  bool flat = false;
};
constexpr int kSpanBS = 512;
constexpr int kSpanUnroll = 8;
constexpr int kLaneBS = 256;
constexpr uint64_t kLaneItems = 32768;
// Lanes per block.  Blocks of 256 put a wave on each SIMD of their CU; where they leave a sparse second
// round, single waves spread more evenly: (72, 300000) f32 sum, 75000 lanes, 18.6 -> 16.0 us; but (1000,
// 200003), 50001 lanes, 119 -> 136 and (4000, 100, 300), 300000 lanes, 82 -> 90.
inline uint32_t lane_block(uint64_t items) {
  const uint64_t blocks = ceil_div(items, uint64_t(kLaneBS)), rounds = ceil_div(blocks, uint64_t(256));
  return rounds > 1 && items < 6 * kLaneItems && 100 * blocks < 85 * 256 * rounds ? 64 : kLaneBS;
}
constexpr uint64_t kSpanRowBytes = 4096;
constexpr uint64_t kSpanBlocks = 256;
constexpr uint64_t kSpanStripBytes = uint64_t(4) << 20;

// columns per strip of a small input, 0 for tiles along the rows
inline uint64_t span_strip(uint64_t outer, uint64_t R, uint64_t C, uint64_t es, uint64_t V, uint64_t round) {
  if (C % V != 0 || outer >= kSpanBlocks || R * C <= round || outer * R * C * es > kSpanStripBytes) return 0;
  uint64_t cw = C / ceil_div(kSpanBlocks, outer) / V * V;
  const uint64_t least = 64 / es;  // 64-byte runs
  if (cw < least) cw = least;
  return cw < C && 2 * R * cw <= 3 * round ? cw : 0;
}

enum class RedKind { kSum, kComplexSum, kOrdered };  // sum / prod / mean, of complex elements, max / min / arg

inline ColRoute col_route(const ReducePlan& p, size_t es, RedKind kind) {
  const bool ordered = kind == RedKind::kOrdered;
  ColRoute r;
  const uint32_t V = es >= 16 ? 1 : uint32_t(16 / es);
  const uint64_t C = p.oshape[p.ond - 1], R = p.R;
  const uint64_t outer = p.out_size / C;
  if (p.kind != kColReduce || R >= (uint64_t(1) << 31) || C >= (uint64_t(1) << 31)) return r;
  // the outer dims are decoded in 32 bits
  if (outer >= (uint64_t(1) << 31)) return r;
  const uint64_t vecs = ceil_div(C, V), groups = ceil_div(vecs, 64), items = outer * vecs;
  const bool narrow = vecs <= 16;                     // a quarter of a column group's lanes at most
  const bool part = 10 * vecs <= 6 * 64 * groups;     // 60% of them
  const bool full = 10 * vecs >= 9 * 64 * groups;     // 90%
  // rounds that the column kernel does not fill (its ordered rounds are 32 rows)
  const bool brief = R < (ordered && (es < 8 || part) ? 64 : 25) && (!ordered || part || R % 32 != 0);
  const bool ragged = C % V != 0;  // rows start anywhere: (1000, 200003) f32 sum 147 us by columns, 120 by lanes
  if (C >= V && items < (uint64_t(1) << 31) &&
      ((items >= kLaneItems && (narrow || (ordered && brief) || (ragged && full))) ||
       (items >= 2 * kLaneItems && (brief || (full && (kind != RedKind::kComplexSum || items >= 4 * kLaneItems)))) ||
       items >= 8 * kLaneItems)) {
    r.kind = ColRoute::kLanes;
    return r;
  }
  const uint64_t row = C * es;
  if (row > kSpanRowBytes || (ordered && row == kSpanRowBytes)) return r;
  const bool contiguous = p.rstride == int64_t(C);
  if ((C % V != 0 && !contiguous) || R * C < V) return r;
  const uint64_t round = uint64_t(kSpanBS) * kSpanUnroll * V;  // elements of one round of a whole block
  uint64_t cw = span_strip(outer, R, C, es, V, round);
  if (cw == 0) {
    const uint64_t blocks = outer * groups;  // of the column kernel, before it splits the rows
    bool span;
    if (R * C <= round && blocks <= 128)
      span = true;  // one masked round
    else if (R <= 24)
      span = ordered || narrow;
    else if (blocks <= 24)
      span = ordered ? outer > 1 || (R >= 20000 && (narrow || (vecs % 64 != 0 && R * row >= (uint64_t(64) << 20))))
                     : R >= (kind == RedKind::kComplexSum ? 500 : 1400) || (narrow && outer * R >= 8000);
    else if (narrow)
      span = true;
    else if (R <= 128)
      span = ordered ? row <= 2048 && blocks <= 512 : row <= 1536 && blocks <= (kind == RedKind::kSum ? 128 : 255);
    else if (blocks < 64) {
      // tiles of the column kernel that leave some CUs a second one
      const bool uneven = row >= 1700 && blocks * ceil_div(uint64_t(256), blocks) > 256;
      if (ordered)
        span = part || (R <= 200 ? row <= 2048 : R <= 600 || uneven);
      else if (kind == RedKind::kComplexSum)
        span = row <= 2048 || (R >= 500 && uneven);
      else
        span = (part && R <= 280) || (R >= 700 && uneven);
    } else if (kind == RedKind::kComplexSum)  // (two tiles of 128 to 255 blocks would not fit a stream's workspace)
      span = row <= 2048 || (blocks >= 128 && blocks < 256);
    else
      span = R >= (ordered ? 250 : 500) && blocks >= 64 && blocks <= 512 &&
             (part || (ordered && row <= 2048 && vecs % 64 != 0));
    if (!span) return r;
    cw = C;
  }
  const uint32_t period = uint32_t(cw) / gcd32(uint32_t(cw), V);  // lanes of the shortest whole-row step
  if (period > uint32_t(kSpanBS)) return r;
  r.cw = uint32_t(cw);
  r.strips = uint32_t(ceil_div(C, cw));
  if (outer * r.strips * kSpanBlocks >= (uint64_t(1) << 31)) return r;
  r.kind = ColRoute::kSpans;
  r.flat = contiguous && r.strips == 1;
  // the block size with the fewest idle lanes, no larger than one round of the slice needs
  uint64_t most = ceil_div(ceil_div(R * cw, uint64_t(V) * kSpanUnroll), 64) * 64;
  const uint64_t least = ceil_div(period, 64) * 64;
  if (most < least) most = least;
  if (most > uint64_t(kSpanBS)) most = kSpanBS;
  for (uint32_t bs = uint32_t(most); bs >= least && 2 * bs > most; bs -= 64) {
    const uint32_t n = bs / period * period;
    if (r.bs == 0 || uint64_t(n) * r.bs > uint64_t(r.lanes) * bs + uint64_t(r.bs) * bs / 50) {
      r.bs = bs;
      r.lanes = n;
    }
  }
  r.m = uint32_t(uint64_t(r.lanes) * V / cw);
  // 256 blocks, one per CU with 8 x 16-byte loads in flight per lane, twice buffered ((1000003, 37) f32
  // mean 30.8 us, 32.8 with 512 and 36.2 with 1024).  A second launch folds the tiles: not worth it
  // below 6 rounds
  const uint64_t chunks = R / (uint64_t(r.m) * kSpanUnroll);
  uint64_t tiles = ceil_div(kSpanBlocks, outer * r.strips);
  if (tiles > chunks / 2) tiles = chunks / 2;
  // the partials (at most 2 * es bytes each) have to fit the 1 MiB workspace of a stream
  const uint64_t room = (uint64_t(1) << 20) / (p.out_size * 2 * es);
  if (tiles > room) tiles = room;
  r.tiles = uint32_t(chunks < 6 || tiles < 1 ? 1 : tiles);
  return r;
}

// ---------------------------------------------------------------------------------------------
// Row lengths that the short-row kernel, whose groups are powers of two, leaves to the kernels with 16
// lanes or one lane per row: accumulators of more than 8 bytes (two rows in flight per group instead
// of four) whose rows leave almost half of a group idle.  Its time against theirs, 6M and 40M elements:
// c64 sums of 33 1.31 and 1.39, of 50 1.0 and 1.05; f64 max of 33 1.12 and 1.19, of 40 1.10 and 1.12, of 5
// 1.06 and 1.0; f64 sums of 33 and 40 (8 bytes) 0.86 and 0.85, 0.82 and 0.76.
inline bool short_rows_pay(uint64_t R, uint64_t vecs, size_t acc_bytes, bool ordered) {
  if (acc_bytes <= 8) return true;
  return !(ordered && R == 5) && (vecs <= 16 || vecs > (ordered ? 24u : 26u));
}

// ---------------------------------------------------------------------------------------------
// Max / min / arg over segments of 16 KB and more: a wave per segment instead of a 512-lane block.  The few
// elements per lane of a block improve the running extreme in nearly every chunk, and each time cost the
// search for its index, so waves win while a segment is short and there are enough of them for all CUs:
// (16384, 4096) f32 max 65 us by blocks, 42 by waves; (2048, 4096) 1.24 times as fast by waves, (1024,
// 4096) 1.05, (1024, 4500) 0.94, (500, 6000) 0.74, (64, 8000) 0.60; (2048, 8000) 1.06, (16384, 8000) 0.92.
inline bool ordered_waves(uint64_t seg_bytes, uint64_t segments) {
  if (seg_bytes < 16384 || seg_bytes >= 32768) return false;
  return segments >= (seg_bytes <= 17408 ? 768 : 1536) && (seg_bytes <= 28672 || segments < 5000);
}

// ---------------------------------------------------------------------------------------------
// Which loads of a large elementwise op stream (elementwise.hip).
constexpr uint64_t kLine = 128;

// distinct elements operand `o` of a plan reads (broadcast dims, stride 0, count once)
inline uint64_t operand_elems(const Plan& p, int o) {
  uint64_t n = 1;
  for (int d = 0; d < p.ndim; ++d)
    if (p.stride[o][d] != 0) n *= p.shape[d];
  return n;
}

// true when every row that operand `o` walks starts on a multiple of `unit` bytes
inline bool rows_at(const Plan& p, int o, const void* ptr, size_t es, uint64_t unit) {
  uintptr_t q = reinterpret_cast<uintptr_t>(ptr);
  for (int d = 0; d < p.ndim; ++d) {
    const int64_t s = p.stride[o][d];
    if (s == -1) q -= (p.shape[d] - 1) * es;  // a flipped row starts at its far end
    if (s < -1 || s > 1)
      if ((s < 0 ? uint64_t(-s) : uint64_t(s)) * es % unit) return false;
  }
  return q % unit == 0;
}

// whether the address ranges of operands 1 and 2 meet
inline bool operands_meet(const Plan& p, const void* a, const void* b, size_t es) {
  int64_t lo[2] = {0, 0}, hi[2] = {0, 0};
  for (int d = 0; d < p.ndim; ++d)
    for (int k = 0; k < 2; ++k) {
      const int64_t e = p.stride[k + 1][d] * int64_t(p.shape[d] - 1);
      (e < 0 ? lo : hi)[k] += e;
    }
  const int64_t pa = int64_t(reinterpret_cast<intptr_t>(a)), pb = int64_t(reinterpret_cast<intptr_t>(b));
  const int64_t n = int64_t(es);
  return pa + lo[0] * n <= pb + hi[1] * n && pb + lo[1] * n <= pa + hi[0] * n;
}

// Which operands of a large binary op stream: those read once, each by itself; a broadcast one does not,
// and does not decide for the other.  Rows that start inside a line share their first and last line with
// their neighbours, and a streamed line is not kept for them; that only shows where the kernel reads more
// than these rows and the output: beside a broadcast row, and where the other operand walks the same
// lines.  Rotated buffers, default against streaming loads, f32 and f64: x - row of (8009, 4003) 46 against
// 49 us, of (20000, 3000) f64 196 against 213; neighbours along rows of 4003 f64 90 against 106; but x -
// column at any address 110 against 103 and 220 against 206 at (20000, 4096), two slices of rows of 4100
// 137 against 124 and 271 against 251, one flat operand 16 bytes off a line 135 against 126 and 136 against
// 126 at 256 MB each, x times a scalar anywhere 84 against 80.
// Tiles of a transposed operand read parts of many rows and stream only where every row that is not broadcast
// starts on a line (the sum with a transposed (8192, 4096) view 71 us streamed, 75 by default).
struct LoadPolicy { bool a, b, tiles; };
inline LoadPolicy binary_loads(const Plan& p, const void* a, const void* b, size_t es, bool big) {
  if (!big) return LoadPolicy{false, false, false};
  const bool one = operand_elems(p, 1) == p.numel, two = operand_elems(p, 2) == p.numel;
  const int L = p.ndim - 1;
  auto row = [&](int o) { return p.ndim > 1 && p.stride[o][L] != 0 && operand_elems(p, o) < p.numel; };
  const bool off_a = one && !rows_at(p, 1, a, es, kLine), off_b = two && !rows_at(p, 2, b, es, kLine);
  bool shared = false;
  if (off_a) shared = row(2) || (two && operands_meet(p, a, b, es));
  if (off_b) shared = shared || row(1) || (one && operands_meet(p, a, b, es));
  return LoadPolicy{one && !shared, two && !shared, !off_a && !off_b};
}

// ---------------------------------------------------------------------------------------------
// The tile of a binary op whose transposed operand is P x L per matrix (elementwise.hip), or none: the
// row kernels gather the operand from the caches.  P and L below 16 would leave a tile mostly empty.
// With L of up to 32 even the tall tile is mostly empty when P is short too, and the row kernels win once
// they fill the GPU.  Sums by rows, tall and small tiles (us):
//  * below 4 to 12 MB any tile beats the rows: (750, 20, 20) f32 9.0, 5.2 and 3.9; in 16-byte elements
//    (938, 20, 16) 8.0, 5.7 and 7.1, (625, 20, 24) 7.9, 5.9 and 5.8;
//  * up to 64 MB the tall tile needs a long P ((4500, 100, 20) f32 35.1 by rows, 29.6 tall; f64 40.7 and 44.6,
//    so 8-byte elements only up to 48 MB), the small one 32 rows ((8789, 32, 32) f32 34.6, 23.6 small);
//  * beyond, and from 10 MB in 16 bytes, the rows win ((78125, 16, 16) f32 46, 220 and 92; (12500, 100, 16) 47
//    and 65 tall) or are level, but for 4-byte matrices that fill a good part of a tall tile: (4883, 128, 32)
//    51.9 and 44.0, (300, 5000, 17) 101 and 66.
enum class BinTile { kNone, kTall, kSmall, kLarge };
inline BinTile binary_tile(uint64_t P, uint64_t L, uint64_t numel, size_t es) {
  if (P < 16 || L < 16) return BinTile::kNone;
  if (L > 32) return L <= 64 || P <= 64 || numel < (uint64_t(4) << 20) ? BinTile::kSmall : BinTile::kLarge;
  const uint64_t mb = numel * es >> 20;
  if (es >= 16) return mb >= 10 ? BinTile::kNone : L <= 20 ? BinTile::kTall : BinTile::kSmall;
  const bool tall = P >= (es == 4 ? 100 : 64);
  if (mb < (tall ? 4 : P * L < 1024 ? 10 : 12)) return BinTile::kSmall;
  if (mb >= 64) return es == 4 && L > 16 && P * L >= 3072 ? BinTile::kTall : BinTile::kNone;
  if (tall && (es == 4 || mb < 48)) return BinTile::kTall;
  return L >= 30 && P >= (es == 4 ? 24 : 32) ? BinTile::kSmall : BinTile::kNone;
}

// ---------------------------------------------------------------------------------------------
// How a scan of a strided axis with unit-stride columns runs (scan.hip).
//
// Tiles: 16 lanes across (256-byte runs) by 512 lanes of 8 rows, so 256 rows.  The few strips of a
// narrow array cannot keep the 8 XCDs equally busy under that block numbering, so below 32 strips,
// where their count is not a multiple of 8, tiles are claimed from a counter instead (their
// predecessors are then running or finished on whatever XCD), in 512-row tiles of 1024 lanes, which
// halve the look-backs.  Fewer columns than a 16-byte vector holds take 4 lanes across, one column
// each.
//
// One lane per column keeps the order of the reference, with 32 rows of loads in flight (`depth`):
// axes of 64 to 384 rows ((300, 20000) f32 26.8 -> 13.9 us; (380, 500) 28.4 -> 14.1), and longer ones
// of many slices whose rows leave most of a tile's columns idle ((10000, 500, 5) f32 159 us by tiles, 90 by
// lanes; (50000, 500, 2) 588 and 225; (10000, 1000, 3) f64 350 and 180).  From 512 KB per row of the
// output on there are lanes enough for longer axes too, with 16 rows in flight ((1000, 131072) f32 184 us, 210 in
// tiles; (1000, 65536) f64 184 and 209) or, where a row is at most 64 bytes, 32 ((50000, 390, 5) f32 291, 328
// with 16).
//
// kNone, one lane per column with 4 rows in flight, is enough from 1 MB per row on ((1000, 262144) f32 369 us, 411
// with 16 rows) and from 640 KB on for 8-byte elements and axes below 200 rows ((600, 100000) f64 182 us, 193 with
// 16; (10, 64, 20000) f32 21.9 and 23.6), and is ahead for some short axes: few columns in f32 ((1000,
// 64, 2) 13.4 us against 16.2 with 32, (1000, 100, 5) 13.3 and 15.6; in f64 (1000, 100, 2) is 21.0 and 14.7), and
// rows of 160 bytes and more in f64 ((100, 4096) 9.5 and 10.3).
constexpr int kColLpc = 16, kColLpcThin = 4, kColBlock = 512, kColBlockClaim = 1024, kColRpl = 8;
constexpr uint64_t kColClaimGroups = 32;
constexpr uint64_t kLaneScanRows = 64, kOrderedScanRows = 384;
struct ColScanRoute {
  enum : int { kNone = 0, kLane = 1, kTiles = 2 };
  int kind = kNone;
  uint32_t cols = 0;                       // lane route: lanes
  int depth = 0;                           // lane route: rows of loads in flight, 32 or 16
  bool stream = false;                     // whether a large array may stream
  uint32_t strips = 0, groups = 0, tiles = 0, per = 0;  // per: groups per tile row of the grid
  bool claim = false;
  uint64_t words = 0;                      // tile route: status words (0 for a single tile)

  // Rows that are not whole lines share some with the next row, which other lanes or a later round read, and a
  // streamed line is not kept for them: lanes along rows of 4 KB and more meet few such lines, tiles of 256-byte
  // runs from 256 bytes on or with half lines.  (30000, 100, 7) f32 128 us streamed, 82 by default; rows of
  // 64 bytes, (10000, 390, 8) f64 by lanes, 145 and 134.
  void lane(const ScanPlan& p, size_t es, int rows_ahead) {
    const uint64_t row = p.oshape[p.ond - 1] * es;
    kind = kLane;
    depth = rows_ahead;
    stream = row % kLine == 0 || row >= 4096;
    words = 0;
  }
};

// `acc_words`: status words per column and tile, 1 for 4-byte accumulators, else 2
inline ColScanRoute scan_columns_route(const ScanPlan& p, size_t es, uint64_t acc_words) {
  ColScanRoute r;
  const uint64_t VE = 16 / es;
  const uint64_t C = p.oshape[p.ond - 1];
  if (p.kind != kColScan || C >= (uint64_t(1) << 31) || p.L >= (uint64_t(1) << 40)) return r;
  if (p.rows >= (uint64_t(1) << 31)) return r;
  const uint64_t outer = p.rows / C, row = C * es, kb = p.rows * es >> 10;
  r.cols = uint32_t(p.rows);
  if (p.L < kLaneScanRows || kb >= 1024) return r;
  if (kb >= 512) {
    if (row <= 64) r.lane(p, es, 32);
    else if (row < 512 || kb < 640 || (es == 4 && p.L >= 200)) r.lane(p, es, 16);
    return r;
  }
  const bool thin = C < VE;
  const uint64_t SC = thin ? kColLpcThin : kColLpc * VE;
  const uint64_t strips = (C + SC - 1) / SC;
  if (p.L <= kOrderedScanRows) {
    const bool few = es == 8 ? kb < 48 && row >= 160 && p.L > 64 && p.L <= 112
                             : row < 32 && p.L <= 256 && kb < (p.L < 100 ? 100 : 48);
    if (!few) r.lane(p, es, 32);
    return r;
  }
  r.lane(p, es, 32);
  if (outer >= 5000 && (thin ? p.L <= 512 : strips == 1 && row <= 80)) return r;
  const uint64_t groups = outer * strips;
  const bool claim = thin || (groups < kColClaimGroups && groups % 8 != 0);
  const uint64_t TR = uint64_t(claim ? kColBlockClaim : kColBlock) / (thin ? kColLpcThin : kColLpc) * kColRpl;
  const uint64_t tiles = (p.L + TR - 1) / TR;
  const uint64_t per = claim ? groups : (groups + 7) / 8 * 8;
  if (!grid_fits(per * tiles, claim ? kColBlockClaim : kColBlock)) return r;
  r.kind = ColScanRoute::kTiles;
  r.stream = row % 64 == 0 || row >= 256;
  r.strips = uint32_t(strips);
  r.groups = uint32_t(groups);
  r.tiles = uint32_t(tiles);
  r.per = uint32_t(per);
  r.claim = claim;
  r.words = tiles > 1 || claim ? (claim ? 1 : 0) + groups * tiles * SC * acc_words : 0;
  return r;
}

}  // namespace mpy
