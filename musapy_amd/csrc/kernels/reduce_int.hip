// reduce_int.hip -- reductions of integers narrower than the reference's compute dtype, for gfx950.
//
// The reference casts first (op_builder.rs:2209-2225: integer sums, products and extremes run in
// int64, means in float64) and so does its kernel ABI.  Here the kernels of reduce_kernels.hpp read
// the narrow elements and widen them in registers: the input is read once, at its own width, and
// no wide copy is written.  They stay bound by that read: (4096, 8192) i32 sum over axis 1 105.6 ->
// 23.6 us (5.7 TB/s), argmax 107.2 -> 24.5, mean over axis 0 105.8 -> 27.9, whole-array sum 105.8 ->
// 27.0; (20000, 16384) u8 sum over axis 1 1069 -> 61 us.  Results are those of the cast:
//   sum, prod    wrapping 64-bit arithmetic (any order gives the same bits)
//   max, min, arg  compared as 32-bit integers (u32: 64-bit), first index on ties
//   mean         sources of at most 32 bits: the exact 64-bit sum, rounded once to f64 and divided
//                (below 2^53 the float64 sum of the cast is that same integer); 64-bit sources: sums
//                of float64
#include "reduce_kernels.hpp"

namespace mpy {
namespace {

// elements per 16-byte load, at most 8 (1-byte elements move 8 bytes: 16 wide accumulators and
// their unrolled loads would not fit the registers)
template <class S> constexpr int ivec() { return sizeof(S) == 1 ? 8 : int(16 / sizeof(S)); }

struct IntCall {
  int ndim;
  const size_t* shape;
  const ssize_t* strides;
  int axis;
  size_t axis_len, out_size;
  void* tmp;
  size_t tmp_bytes;
  hipStream_t st;
};

// How a call runs: one lane per output vector, spans of rows (strided axis, unit-stride outputs), or
// row segments.  `tiles` > 1: partials in tmp, folded by a second launch.
struct IntRoute {
  enum : int { kRows = 0, kLanes = 1, kSpans = 2 };
  int kind = kRows;
  ColRoute span;
  size_t tiles = 1;
};

IntRoute int_route(const ReducePlan& p, size_t es, uint32_t V) {
  IntRoute r;
  const uint64_t C = p.oshape[p.ond - 1];
  const uint64_t outer = p.out_size / C;
  if (p.kind == kColReduce && C >= V) {
    if (outer * ceil_div(C, V) >= kLaneItems) {
      r.kind = IntRoute::kLanes;
      return r;
    }
    r.kind = IntRoute::kSpans;
    ColRoute& s = r.span;
    const bool contiguous = p.rstride == int64_t(C);
    uint64_t cw = C;
    // whole contiguous rows where a block holds their period, else strips of 128 lanes
    if (!contiguous || C * es > kSpanRowBytes / 2 || C / gcd32(uint32_t(C), V) > uint32_t(kSpanBS)) {
      cw = uint64_t(V) * 128;
      const uint64_t all = ceil_div(C, V) * V;
      if (cw > all) cw = all;
    }
    const uint64_t round = uint64_t(kSpanBS) * kSpanUnroll * V;
    if (outer < kSpanBlocks && p.R * C > round && outer * p.R * C * es <= kSpanStripBytes) {
      // small inputs: strips instead of tiles, one launch (see col_route)
      uint64_t per = C / ceil_div(kSpanBlocks, outer) / V * V;
      const uint64_t least = 64 / es;
      if (per < least) per = least;
      if (per < cw) cw = per;
    }
    s.cw = uint32_t(cw);
    s.strips = uint32_t(ceil_div(C, cw));
    s.flat = contiguous && cw == C;
    const uint32_t period = uint32_t(cw) / gcd32(uint32_t(cw), V);
    s.bs = kSpanBS;
    s.lanes = kSpanBS / period * period;
    s.m = uint32_t(uint64_t(s.lanes) * V / cw);
    const uint64_t chunks = p.R / (uint64_t(s.m) * kSpanUnroll);
    uint64_t tiles = ceil_div(kSpanBlocks, outer * s.strips);
    if (tiles > chunks / 2) tiles = chunks / 2;
    s.tiles = uint32_t(chunks < 6 || tiles < 1 ? 1 : tiles);
    r.tiles = s.tiles;
    return r;
  }
  // row segments: as tiles_hint, for segments of at least 32 KB
  if (p.out_size < 2048 && p.out_size * p.R * es > (uint64_t(128) << 10)) {
    uint64_t tiles = ceil_div(uint64_t(4096), p.out_size);
    const uint64_t most = ceil_div(p.R * es, 32768);
    r.tiles = size_t(tiles < most ? tiles : most);
    if (r.tiles < 1) r.tiles = 1;
  }
  return r;
}

bool int_plan(ReducePlan& p, const IntCall& c) {
  if (c.out_size == 0 || c.axis_len == 0 || !args_ok(c.ndim, c.axis)) return false;
  plan_reduce(p, c.ndim, c.shape, c.strides, c.axis, c.axis_len, c.out_size);
  return p.R < (uint64_t(1) << 31) && c.out_size < (uint64_t(1) << 31);
}

template <class Op, class T, class S, class O, int WRITE>
void launch_int_rows(const S* a, RedOut<O> out, const ReducePlan& p, size_t tiles, hipStream_t st) {
  constexpr int V = ivec<S>();
  if constexpr (WRITE == kWriteFinal) {
    if (tiles == 1 && launch_short<Op, T, V, S, O>(a, out, p, st)) return;
  }
  RowArgs ra{};
  ra.ix = out_indexer(p, p.ond);
  ra.R = p.R;
  ra.rs = p.rstride;
  ra.tiles = uint32_t(tiles);
  ra.chunk = ceil_div(ceil_div(p.R, tiles), uint64_t(V)) * V;
  ra.nwork = p.out_size * tiles;
  const bool vec = p.rstride == 1;
  const uint64_t seg = ra.chunk < p.R ? ra.chunk : p.R;
  if (seg * sizeof(S) >= 16384) {  // (8192, 8192) u8 in 8 KB rows: 25.2 us by blocks, 14.6 by waves
    const unsigned grid = unsigned(ra.nwork);
    if (vec) k_reduce_row<Op, T, kRowBS, kRowBS, V, 4, WRITE, S, O><<<grid, kRowBS, 0, st>>>(a, ra, out);
    else k_reduce_row<Op, T, kRowBS, kRowBS, 1, 8, WRITE, S, O><<<grid, kRowBS, 0, st>>>(a, ra, out);
  } else if (seg >= 64) {
    const unsigned grid = unsigned(ceil_div(ra.nwork, kRBlock / kWave));
    if (vec) k_reduce_row<Op, T, kRBlock, kWave, V, 2, WRITE, S, O><<<grid, kRBlock, 0, st>>>(a, ra, out);
    else k_reduce_row<Op, T, kRBlock, kWave, 1, 4, WRITE, S, O><<<grid, kRBlock, 0, st>>>(a, ra, out);
  } else if (seg >= 8 && vec) {
    const unsigned grid = unsigned(ceil_div(ra.nwork, kRBlock / 16));
    k_reduce_row<Op, T, kRBlock, 16, 1, 2, WRITE, S, O><<<grid, kRBlock, 0, st>>>(a, ra, out);
  } else {
    const unsigned grid = unsigned(ceil_div(ra.nwork, kRBlock));
    k_reduce_row<Op, T, kRBlock, 1, 1, 4, WRITE, S, O><<<grid, kRBlock, 0, st>>>(a, ra, out);
  }
}

// Op: the streaming fold over T; OpF: the fold of arg partials (absolute indices); O: what is written
template <class Op, class OpF, class T, class S, class O>
int run_int(const void* av, RedOut<O> out, const IntCall& c) {
  constexpr int V = ivec<S>();
  const S* a = static_cast<const S*>(av);
  ReducePlan p;
  if (!int_plan(p, c)) return -1;
  IntRoute r = int_route(p, sizeof(S), V);
  const uint64_t C = p.oshape[p.ond - 1];
  if (r.kind == IntRoute::kLanes) {
    const uint32_t vpr = uint32_t(ceil_div(C, V));
    const uint32_t items = uint32_t(p.out_size / C * vpr);
    const uint32_t bs = lane_block(items);
    k_reduce_lane<Op, T, V, kSpanUnroll, S, O><<<dim3(unsigned(ceil_div(items, bs))), bs, 0, c.st>>>(
        a, out_indexer(p, p.ond - 1), uint32_t(C), make_fastdiv(vpr), p.R, p.rstride, items, out);
    return 0;
  }
  if (r.kind == IntRoute::kSpans) {
    using A = typename Op::A;
    SpanArgs sa{};
    sa.ix = out_indexer(p, p.ond - 1);
    sa.C = uint32_t(C);
    sa.cw = r.span.cw;
    sa.strips = r.span.strips;
    sa.m = r.span.m;
    sa.lanes = r.span.lanes;
    sa.R = p.R;
    sa.rs = p.rstride;
    sa.whole = uint32_t(p.R / (uint64_t(r.span.m) * kSpanUnroll));
    sa.flat = r.span.flat;
    const uint64_t outer = p.out_size / C;
    const bool room = c.tmp != nullptr && c.tmp_bytes >= p.out_size * r.tiles * sizeof(A);
    sa.tiles = r.tiles > 1 && room ? uint32_t(r.tiles) : 1;
    const dim3 grid(unsigned(outer * sa.strips * sa.tiles));
    A* part = static_cast<A*>(c.tmp);
    if (sa.tiles == 1) {
      k_reduce_span<Op, T, V, kSpanUnroll, true, S, O><<<grid, r.span.bs, 0, c.st>>>(a, sa, out, part);
      return 0;
    }
    k_reduce_span<Op, T, V, kSpanUnroll, false, S, O><<<grid, r.span.bs, 0, c.st>>>(a, sa, out, part);
    const uint32_t cb = C < 32 ? uint32_t(C) : 32;
    const uint32_t groups = uint32_t(ceil_div(C, cb));
    k_span_final<Op, T, S, O><<<dim3(unsigned(outer * groups)), kSpanBS, 0, c.st>>>(a, part, sa.ix, sa.C, sa.tiles, cb,
                                                                                groups, out);
    return 0;
  }
  const size_t per = sizeof(T) + (Op::kArg ? 8 : 0);
  if (r.tiles > 1 && (c.tmp == nullptr || c.tmp_bytes < p.out_size * r.tiles * per)) r.tiles = 1;
  if (r.tiles == 1) {
    launch_int_rows<Op, T, S, O, kWriteFinal>(a, out, p, 1, c.st);
    return 0;
  }
  const size_t n = p.out_size * r.tiles;
  if constexpr (Op::kArg) {
    int64_t* pi = static_cast<int64_t*>(c.tmp);
    T* pv = reinterpret_cast<T*>(pi + n);
    launch_int_rows<Op, T, S, T, kWritePair>(a, RedOut<T>{pv, pi, 0.0, kFinPlain}, p, r.tiles, c.st);
    launch_pairs<OpF, T, kWriteFinal>(pv, pi, RedOut<T>{nullptr, out.idx, 0.0, kFinPlain}, r.tiles, p.out_size, 1, c.st);
  } else {
    T* pv = static_cast<T*>(c.tmp);
    launch_int_rows<Op, T, S, T, kWriteVal>(a, RedOut<T>{pv, nullptr, 0.0, kFinPlain}, p, r.tiles, c.st);
    const size_t shape[2] = {p.out_size, r.tiles};
    const ssize_t strides[2] = {ssize_t(r.tiles), 1};
    ReducePlan q;
    plan_reduce(q, 2, shape, strides, 1, r.tiles, p.out_size);
    launch_int_rows<Op, T, T, O, kWriteFinal>(pv, out, q, 1, c.st);
  }
  return 0;
}

template <class S>
int int_values(int op, const void* a, void* cv, const IntCall& c) {
  // extremes compare as the narrowest of int32 / int64 that holds S
  using K = std::conditional_t<sizeof(S) < 4 || std::is_same_v<S, int32_t>, int32_t, int64_t>;
  const RedOut<int64_t> val{static_cast<int64_t*>(cv), nullptr, 0.0, kFinPlain};
  const RedOut<int64_t> idx{nullptr, static_cast<int64_t*>(cv), 0.0, kFinPlain};
  switch (op) {
    case MUSAPY_RED_SUM: return run_int<OpSum<int64_t>, OpSum<int64_t>, int64_t, S>(a, val, c);
    case MUSAPY_RED_PROD: return run_int<OpProd<int64_t>, OpProd<int64_t>, int64_t, S>(a, val, c);
    case MUSAPY_RED_MAX: return run_int<OpExt<K, true, false>, OpExt<K, true, false>, K, S>(a, val, c);
    case MUSAPY_RED_MIN: return run_int<OpExt<K, false, false>, OpExt<K, false, false>, K, S>(a, val, c);
    case MUSAPY_RED_ARGMAX: return run_int<OpExt<K, true, true>, OpExt<K, true, true, int64_t>, K, S>(a, idx, c);
    case MUSAPY_RED_ARGMIN: return run_int<OpExt<K, false, true>, OpExt<K, false, true, int64_t>, K, S>(a, idx, c);
    case MUSAPY_RED_MEAN: {
      const RedOut<double> mean{static_cast<double*>(cv), nullptr, mean_count<double>(c.axis_len), kFinMean};
      return run_int<OpSum<int64_t>, OpSum<int64_t>, int64_t, S>(a, mean, c);
    }
  }
  return -1;
}
// 64-bit sources: only the mean is cast (to f64)
template <class S>
int int_mean64(int op, const void* a, void* cv, const IntCall& c) {
  if (op != MUSAPY_RED_MEAN) return -1;
  const RedOut<double> mean{static_cast<double*>(cv), nullptr, mean_count<double>(c.axis_len), kFinMean};
  return run_int<OpSum<double>, OpSum<double>, double, S>(a, mean, c);
}

template <class S>
size_t int_scratch(int op, const IntCall& c) {
  ReducePlan p;
  if (!int_plan(p, c)) return 0;
  const IntRoute r = int_route(p, sizeof(S), ivec<S>());
  if (r.tiles <= 1) return 0;
  return p.out_size * r.tiles * 16;  // an accumulator, or a value and an index: at most 16 bytes
}

}  // namespace
}  // namespace mpy

using namespace mpy;

extern "C" {

size_t musapy_reduce_int_scratch_v1(int op, int src_dtype, int ndim, const size_t* in_shape, const ssize_t* in_strides,
                                    int axis, size_t axis_len, size_t out_size) {
  const IntCall c{ndim, in_shape, in_strides, axis, axis_len, out_size, nullptr, 0, nullptr};
  switch (src_dtype) {
    case MUSAPY_DT_I8: case MUSAPY_DT_U8: return int_scratch<int8_t>(op, c);
    case MUSAPY_DT_I16: case MUSAPY_DT_U16: return int_scratch<int16_t>(op, c);
    case MUSAPY_DT_I32: case MUSAPY_DT_U32: return int_scratch<int32_t>(op, c);
    case MUSAPY_DT_I64: case MUSAPY_DT_U64: return int_scratch<int64_t>(op, c);
  }
  return 0;
}

int musapy_reduce_int_v1(int op, int src_dtype, const void* a, void* c, int ndim, const size_t* in_shape,
                         const ssize_t* in_strides, int axis, size_t axis_len, size_t out_size, void* tmp,
                         size_t tmp_bytes, hipStream_t st) {
  const IntCall k{ndim, in_shape, in_strides, axis, axis_len, out_size, tmp, tmp_bytes, st};
  switch (src_dtype) {
    case MUSAPY_DT_I8: return int_values<int8_t>(op, a, c, k);
    case MUSAPY_DT_I16: return int_values<int16_t>(op, a, c, k);
    case MUSAPY_DT_I32: return int_values<int32_t>(op, a, c, k);
    case MUSAPY_DT_U8: return int_values<uint8_t>(op, a, c, k);
    case MUSAPY_DT_U16: return int_values<uint16_t>(op, a, c, k);
    case MUSAPY_DT_U32: return int_values<uint32_t>(op, a, c, k);
    case MUSAPY_DT_I64: return int_mean64<int64_t>(op, a, c, k);
    case MUSAPY_DT_U64: return int_mean64<uint64_t>(op, a, c, k);
  }
  return -1;
}

}  // extern "C"
