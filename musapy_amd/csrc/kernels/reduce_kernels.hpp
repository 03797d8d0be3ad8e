// reduce_kernels.hpp -- sum / prod / max / min / mean / argmax / argmin over one axis, for gfx950.
//
// Drop-in for the reference's kernels/reduction.mu:1342-2055 (the `_v2` wrappers: naive,
// small_axis, partial, final, mid).  All entry points share two streaming kernels chosen from
// the host plan (plan.hpp):
//   row  the reduced axis is the walk direction: a group of lanes (a whole block, one wave, or a
//        single lane for very short axes) reduces one (output, tile) segment with 16-byte loads
//        when the axis is unit-stride, then combines through wave-64 butterflies and LDS;
//   col  the reduced axis is strided but the innermost output dim is unit-stride (axis=0 of a
//        C-order matrix): 64 lanes x VEC walk adjacent columns, the 4 waves of a block split the
//        rows, and LDS merges the waves -- every load is a coalesced row segment.  Narrow rows
//        take whole rows per step instead (span kernel), and reductions with many outputs one
//        lane per 16 bytes of them (lane kernel); col_route holds the lines between the three.
// Reductions write next to nothing, so their loads stream at every volume measured (the 128 MB c64
// sum: 5.1 TB/s, 4.6 with default loads).  Large reductions are split into tiles: the partial entry points write [out_size][tiles] and
// the final entry points reduce those rows with the same row kernel.  Every combine order is
// fixed, so results are identical from run to run.
#pragma once

#include "kcommon.hpp"
#include "reduce_ops.hpp"
#include "routes.hpp"
#include "publish.hpp"
#include "../../../include/musapy_kernels.h"

#include <atomic>
#include <type_traits>
#include <mutex>

namespace mpy {

constexpr int kRBlock = 256;
constexpr int kRowBS = 512;  // block size of the block-per-segment row kernel (measured best on MI355X)
// Whole-array reductions: 256-lane blocks, each lane keeping 8 x 16-byte loads in flight (32 KB
// chunks).  At a quarter of the waves of 512-lane blocks with 4 loads per lane, a 64M f32 sum with
// its hand-over measured 40.5 us event-timed against 41.4-41.5 us (a one-round grid of 1024
// blocks; 2048 blocks 40.9 us, 4096 blocks 41.5-42.1 us): the 8192 waves of the previous grid
// took the dispatcher about 3.6 us to start.
constexpr int kAllBS = 256;
constexpr int kAllUnroll = 8;
// Chunks of loads held per lane (walk_chunks): kAllBuffers - 1 chunks in flight at each fold.  With
// the same registers, 4 buffers of 4 loads (12 in flight at each fold) and 3 of 4 measured no faster
// than 2 of 8 (64M f32 sum, argmax and max over (0,1) within 0.5 us, 256M level): the folds are not
// what holds the stream back.
constexpr int kAllBuffers = 2;

// what a kernel writes per (output, tile)
enum : int { kWriteFinal = 0, kWriteVal = 1, kWritePair = 2 };
// which final transform applies to an additive accumulator
enum : int { kFinPlain = 0, kFinMean = 1 };

template <class T>
struct RedOut {
  T* val;            // final values (kWriteFinal of value ops) or partial values
  int64_t* idx;      // arg results (kWriteFinal of arg ops) or partial indices
  double count;      // mean divisor
  int fin;
};

// --------------------------------------------------------------------------------------------
// Writing one finished accumulator.
// O: the element type written (T, except where a reduction of narrow integers widens its result).
template <class Op, class T, int WRITE, class O = T>
__device__ inline void write_result(const RedOut<O>& out, uint64_t slot, typename Op::A acc, int64_t k0 = 0) {
  if constexpr (Op::kOrdered) {
    if constexpr (WRITE == kWritePair) {
      out.val[slot] = acc.idx < 0 ? T(0) : acc.val;
      out.idx[slot] = acc.idx < 0 ? int64_t(-1) : k0 + int64_t(acc.idx);
    } else if constexpr (Op::kArg) {  // final arg result
      out.idx[slot] = acc.idx < 0 ? 0 : k0 + int64_t(acc.idx);
    } else {
      // value max/min: an empty tile writes a marker the next level skips
      if (acc.idx < 0)
        out.val[slot] = Op::better(T(1), T(0)) ? ext_none<T>() : ext_none_min<T>();
      else
        out.val[slot] = acc.val;
    }
  } else {
    if (WRITE == kWriteFinal && out.fin == kFinMean)
      out.val[slot] = mean_of<O>(acc, out.count);
    else
      out.val[slot] = narrow<O>(acc);
  }
}

// NaN at axis position 0 absorbs the whole max/min/arg scan (see reduce_ops.hpp).
template <class Op, class T>
__device__ inline typename Op::A absorb_first(typename Op::A acc, T first) {
  if constexpr (Op::kOrdered) {
    if (is_nan(first)) {
      acc.val = first;
      acc.idx = 0;
    }
  }
  return acc;
}

// --------------------------------------------------------------------------------------------
// f32 max/min accumulators whose indices are below 2^32 - 1 (tile-relative int32, or absolute
// int64 in a whole-array reduction of fewer elements) as one unsigned 64-bit key, so that one
// unsigned max combines two of them instead of Op::comb on (value, index).  The key's high word
// orders the values (sign-magnitude bits mapped to unsigned order, inverted for min) and is never
// 0 for a value; its low word is ~index, so among equal values the lowest index wins, and an empty
// accumulator (key 0) loses to every element.  +0 and -0 compare equal and so share a key (the +0
// bits): whoever decodes a winning zero restores its sign from the element at the winning index.
// Accumulator values are never NaN here (the scan skips NaNs; the NaN-at-position-0 rule is
// applied after the combine), so the result is bit-identical to folding Op::comb.
template <class Op, class I>
__device__ inline uint64_t ext_key_f32(VI<float, I> a) {
  uint32_t u = __builtin_bit_cast(uint32_t, a.val);
  if ((u & 0x7fffffffu) == 0) u = 0;  // -0 -> +0
  u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  if (!Op::kMax) u = ~u;
  return a.idx < 0 ? 0 : (uint64_t(u) << 32) | uint32_t(~uint32_t(a.idx));
}
// the (value, index) of a key; a zero comes back as +0, and key 0 as the empty accumulator
template <class Op, class I>
__device__ inline VI<float, I> ext_unkey_f32(uint64_t key) {
  if (key == 0) return VI<float, I>{0.0f, I(-1)};
  uint32_t v = uint32_t(key >> 32);
  if (!Op::kMax) v = ~v;
  v = (v & 0x80000000u) ? (v & 0x7fffffffu) : ~v;
  return VI<float, I>{__builtin_bit_cast(float, v), I(~uint32_t(key))};
}
// A whole wave's accumulators combined through their keys (one 64-bit max per butterfly step);
// a winning zero takes its sign from the lane that holds the winning index.
template <class Op, class I>
__device__ inline VI<float, I> wave_reduce_ext_f32(VI<float, I> a) {
  uint64_t key = ext_key_f32<Op>(a);
#pragma unroll
  for (int m = kWave / 2; m >= 1; m >>= 1) {
    const uint64_t o = acc_shfl(key, m);
    key = o > key ? o : key;
  }
  VI<float, I> r = ext_unkey_f32<Op, I>(key);
  if (key != 0 && __builtin_bit_cast(uint32_t, r.val) == 0) {
    // a zero won (the same key on every lane): take its sign from its lane
    const bool neg = a.idx == r.idx && (__builtin_bit_cast(uint32_t, a.val) >> 31);
    if (__ballot(neg) != 0) r.val = -0.0f;
  }
  return r;
}

// Group reduction (GROUP lanes -> lane 0 of the group holds the result).  `idx32`: the caller's
// int64 indices are all below 2^32 - 1 and no lane holds a NaN it must keep, so f32 max/min
// accumulators may take the packed-key wave combine (int32 indices always do).
template <class Op, int GROUP>
__device__ inline typename Op::A group_reduce(typename Op::A acc, bool idx32 = false) {
  using A = typename Op::A;
  constexpr bool kKeyed = GROUP >= kWave && Op::kOrdered;
  if constexpr (kKeyed && std::is_same_v<A, VI<float, int32_t>>) {
    acc = wave_reduce_ext_f32<Op>(acc);
  } else if constexpr (kKeyed && std::is_same_v<A, VI<float, int64_t>>) {
    if (idx32) {
      acc = wave_reduce_ext_f32<Op>(acc);
    } else {
#pragma unroll
      for (int m = kWave / 2; m >= 1; m >>= 1) acc = Op::comb(acc, acc_shfl(acc, m));
    }
  } else if constexpr (GROUP > 1) {
    constexpr int W = GROUP < kWave ? GROUP : kWave;
#pragma unroll
    for (int m = W / 2; m >= 1; m >>= 1) acc = Op::comb(acc, acc_shfl(acc, m));
  }
  if constexpr (GROUP > kWave) {
    __shared__ A part[GROUP / kWave];
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    if (lane == 0) part[w] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int i = 1; i < GROUP / kWave; ++i) acc = Op::comb(acc, part[i]);
    }
  }
  return acc;
}

// --------------------------------------------------------------------------------------------
// row kernel: work item w = o * tiles + t, o = output index, t = tile along the axis
struct RowArgs {
  RowIndexer<1> ix;   // output coordinates -> input offset
  uint64_t R;         // axis length
  int64_t rs;         // axis stride
  uint64_t chunk;     // axis elements per tile (multiple of VEC when VEC > 1)
  uint32_t tiles;
  uint64_t nwork;     // out_size * tiles
  bool nt;            // streaming loads; always true: as a run-time value it spaces the loads of WHOLE segments
};

// One lane's share of a segment: lane l of a GROUP-lane group reduces elements l*VEC, l*VEC +
// GROUP*VEC, ... of the n-element segment at tb (indices relative to tb).  tb is unit-stride with
// VEC > 1 (any element address).  S: the stored element, widened to T as it is read.  WHOLE: n is a
// multiple of a round (GROUP * VEC * UNROLL) and tb 16-byte aligned; the loads then test `nt` (always
// true) one by one, and the scalar branches between them leave argmax over the rows of (8192, 8192)
// f32 at 39.9 us, against 41.2 us with the loads back to back.  Lane 0 also returns
// the segment's first element in `first` (ordered reductions need it for the NaN-at-0 rule; it
// is kept from the load instead of being read again at the end).  The fold continues `acc`, and
// ordered reductions record indices as base + (index in the segment).
template <class Op, class T, int GROUP, int VEC, int UNROLL, class S = T, bool WHOLE = false>
__device__ inline typename Op::A accumulate_segment(const S* __restrict__ tb, uint32_t n, int l, int64_t rs,
                                                    T& first, typename Op::A acc = Op::init(),
                                                    int64_t base = 0, bool nt = true) {
  uint32_t k = uint32_t(l) * VEC;
  constexpr uint32_t stepk = uint32_t(GROUP) * VEC;
  const bool lead = l == 0;  // lane 0 starts at element 0
  if (VEC > 1) {
    for (; k + (UNROLL - 1) * stepk + VEC <= n; k += UNROLL * stepk) {
      Vec<S, VEC> x[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        if constexpr (WHOLE) x[u] = vload_pol<S, VEC>(tb + k + u * stepk, nt);
        else x[u] = vload_el<S, VEC>(tb + k + u * stepk);
      }
      // all UNROLL loads are issued before the first use (the scheduler would otherwise hoist
      // arithmetic between them and wait on the first load early)
      __builtin_amdgcn_sched_barrier(0);
      T xs[UNROLL][VEC];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u)
#pragma unroll
        for (int v = 0; v < VEC; ++v) xs[u][v] = T(x[u].v[v]);
      if (Op::kOrdered && lead && k == 0) first = xs[0][0];
      acc = Op::template step_chunk<UNROLL, VEC>(acc, xs, k, stepk, base);
    }
    // The rest in one round of unconditional loads: a vector that the end of the segment cuts is
    // read from where it still fits, and its elements below k (the vector's before) are skipped.
    if (WHOLE) {
    } else if (k < n && n >= uint32_t(VEC)) {
      Vec<S, VEC> x[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const uint32_t ku = k + u * stepk;
        x[u] = vload_el<S, VEC>(tb + (ku + VEC <= n ? ku : n - VEC));
      }
      __builtin_amdgcn_sched_barrier(0);
      if (Op::kOrdered && lead && k == 0) first = T(x[0].v[0]);
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const uint32_t ku = k + u * stepk;
        if (ku + VEC <= n) {
          T xs[1][VEC];
#pragma unroll
          for (int v = 0; v < VEC; ++v) xs[0][v] = T(x[u].v[v]);
          acc = Op::template step_chunk<1, VEC>(acc, xs, ku, 0, base);
        } else if (ku < n) {
#pragma unroll
          for (int v = 0; v < VEC; ++v)
            if (n - VEC + v >= ku) acc = Op::step(acc, T(x[u].v[v]), base + int64_t(n - VEC + v));
        }
      }
    } else {
      for (; k < n; ++k) {  // fewer elements than a vector (lane 0)
        const T x = T(tb[k]);
        if (Op::kOrdered && lead && k == 0) first = x;
        acc = Op::step(acc, x, base + int64_t(k));
      }
    }
  } else {
    for (; k + (UNROLL - 1) * stepk < n; k += UNROLL * stepk) {
      T x[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) x[u] = T(tb[int64_t(k + u * stepk) * rs]);
      if (Op::kOrdered && lead && k == 0) first = x[0];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) acc = Op::step(acc, x[u], base + int64_t(k + u * stepk));
    }
    for (; k < n; k += stepk) {
      const T x = T(tb[int64_t(k) * rs]);
      if (Op::kOrdered && lead && k == 0) first = x;
      acc = Op::step(acc, x, base + int64_t(k));
    }
  }
  return acc;
}

template <class Op, class T, int BS, int GROUP, int VEC, int UNROLL, int WRITE, class S = T, class O = T, bool WHOLE = false>
__global__ __launch_bounds__(BS) void k_reduce_row(const S* __restrict__ a, RowArgs ra, RedOut<O> out) {
  using A = typename Op::A;
  constexpr int kPer = BS / GROUP;  // items per block
  const uint64_t w = uint64_t(blockIdx.x) * kPer + threadIdx.x / GROUP;
  const int l = threadIdx.x % GROUP;
  const bool live = w < ra.nwork;
  A acc = Op::init();
  uint64_t o = 0, t = 0, k0 = 0;
  T first{};
  if (live) {
    // one tile per output (every reduction that fills the GPU with its outputs): no 64-bit
    // division in front of the first load
    if (ra.tiles == 1) {
      o = w;
    } else {
      o = w / ra.tiles;
      t = w - o * ra.tiles;
    }
    int64_t off[1];
    row_offsets<1>(ra.ix, uint32_t(o), off);
    k0 = t * ra.chunk;
    const uint64_t k1 = k0 + ra.chunk < ra.R ? k0 + ra.chunk : ra.R;
    const S* tb = a + off[0] + int64_t(k0) * ra.rs;  // indices below are relative to the tile start
    const uint32_t n = k1 > k0 ? uint32_t(k1 - k0) : 0u;
    acc = accumulate_segment<Op, T, GROUP, VEC, UNROLL, S, WHOLE>(tb, n, l, ra.rs, first, Op::init(), 0, ra.nt);
  }
  acc = group_reduce<Op, GROUP>(acc);
  if (live && (GROUP <= kWave ? l == 0 : threadIdx.x == 0)) {
    if (t == 0 && ra.R > 0) acc = absorb_first<Op, T>(acc, first);
    write_result<Op, T, WRITE, O>(out, w, acc, int64_t(k0));
  }
}

// --------------------------------------------------------------------------------------------
// Fused partial + final for few outputs.  Blocks 0 .. out_size*tiles-1 are the row kernel's
// (output, tile) blocks; each publishes its tile's accumulator (publish.hpp) and exits.  Blocks
// out_size*tiles + o, the last of the grid, are combiners: the dispatcher hands them out after
// every streaming block, so they poll the slots while the last tiles are still streaming and
// finish right after the last publish.  Lane l of a combiner owns tiles l, l + 512, ... (PER of
// them at most, a template parameter so the slot registers do not inflate the streaming blocks'
// register budget), waits until all of them are published (a bounded poll), folds them in
// ascending order, and the block tree combines the lanes: a fixed order, independent of timing.
// A combiner holds one block slot; with at most kFusedMaxOutputs of them the streaming blocks
// always find room, so the waits end.  Every slot read is cleared again, leaving the workspace
// zero.  Workspace: out_size * tiles * W slot words.
constexpr size_t kFusedMaxOutputs = 64;
constexpr size_t kFusedMaxTiles = 2048;  // <= 8 * kRowBS (the largest PER dispatched)
struct FusedArgs {
  uint64_t* slots;
  uint32_t* fault;      // the fault word of the launch's workspace (kcommon.hpp)
  uint32_t spin_limit;  // polls the combiner may make before it gives up
};

// Gathers the published W-word slots lane, lane + kRowBS, ... (below `count`) into v: all
// outstanding slots' words are loaded together, the ready ones kept, the rest polled again.
// Returns false when the poll budget ran out with slots still unpublished.
template <int W, int PER, int STRIDE = kRowBS>
__device__ inline bool gather_published(const uint64_t* slots, uint32_t count, uint32_t spin_limit,
                                        uint64_t (&v)[PER][W]) {
  uint32_t pending = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    if (threadIdx.x + j * STRIDE < count) pending |= 1u << j;
#pragma unroll
    for (int i = 0; i < W; ++i) v[j][i] = 0;
  }
  for (uint32_t spins = 0; pending != 0 && spins < spin_limit; ++spins) {
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (pending & (1u << j))
#pragma unroll
        for (int i = 0; i < W; ++i) v[j][i] = ld_relaxed(slots + uint64_t(threadIdx.x + j * STRIDE) * W + i);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      bool ready = true;
#pragma unroll
      for (int i = 0; i < W; ++i) ready = ready && (v[j][i] & kTag);
      if (ready) pending &= ~(1u << j);
    }
    if (pending) __builtin_amdgcn_s_sleep(2);
  }
  return pending == 0;
}

// After a combiner's gather: true when any lane of the block gave up.  Thread 0 then records the
// fault; the block skips its output write (the caller raises an error instead of returning a
// wrong value).
__device__ inline bool combiner_gave_up(bool ok, uint32_t* fault) {
  const bool bad = __syncthreads_or(ok ? 0 : 1) != 0;
  if (bad && threadIdx.x == 0 && fault) atomicOr(fault, kFaultReduceWait);
  return bad;
}

// a tile's accumulator (tile-relative int32 index) as the final's accumulator (absolute index)
template <class Op, class OpF>
__device__ inline typename OpF::A to_final(const typename Op::A& x, int64_t k0) {
  if constexpr (Op::kOrdered) {
    return typename OpF::A{x.val, x.idx < 0 ? int64_t(-1) : k0 + int64_t(x.idx)};
  } else {
    return x;
  }
}

template <class Op, class OpF, class T, int VEC, int UNROLL, int PER>
__global__ __launch_bounds__(kRowBS) void k_reduce_row_fused(const T* __restrict__ a, RowArgs ra, RedOut<T> out,
                                                             FusedArgs fa) {
  using A = typename Op::A;
  using AF = typename OpF::A;
  static_assert(sizeof(A) % 4 == 0, "accumulator must split into 32-bit slices");
  constexpr int W = int(sizeof(A) / 4);
  const uint64_t w = blockIdx.x;
  if (w < ra.nwork) {  // a streaming (output, tile) block
    const uint64_t o = w / ra.tiles;
    const uint64_t t = w - o * ra.tiles;
    int64_t off[1];
    row_offsets<1>(ra.ix, uint32_t(o), off);
    const uint64_t k0 = t * ra.chunk;
    const uint64_t k1 = k0 + ra.chunk < ra.R ? k0 + ra.chunk : ra.R;
    const uint32_t n = k1 > k0 ? uint32_t(k1 - k0) : 0u;
    T first{};
    A acc = accumulate_segment<Op, T, kRowBS, VEC, UNROLL>(a + off[0] + int64_t(k0) * ra.rs, n, threadIdx.x, ra.rs,
                                                           first);
    acc = group_reduce<Op, kRowBS>(acc);
    if (threadIdx.x == 0) {
      if (t == 0 && ra.R > 0) acc = absorb_first<Op, T>(acc, first);
      uint32_t s[W];
      __builtin_memcpy(s, &acc, sizeof(A));
      publish_slices<W>(fa.slots + w * W, s);
    }
    return;
  }
  // combiner of output o
  const uint64_t o = w - ra.nwork;
  uint64_t* row_slots = fa.slots + o * ra.tiles * W;
  uint64_t v[PER][W];
  const bool ok = gather_published<W, PER>(row_slots, ra.tiles, fa.spin_limit, v);
  AF r = OpF::init();
  A first{};
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t tt = threadIdx.x + j * kRowBS;
    if (tt >= ra.tiles) break;
    uint32_t s[W];
#pragma unroll
    for (int i = 0; i < W; ++i) s[i] = uint32_t(v[j][i]);
    A x;
    __builtin_memcpy(&x, s, sizeof(A));
    if (tt == 0) first = x;
    r = OpF::comb(r, to_final<Op, OpF>(x, int64_t(tt) * int64_t(ra.chunk)));
#pragma unroll
    for (int i = 0; i < W; ++i) st_relaxed(row_slots + uint64_t(tt) * W + i, 0);
  }
  if (combiner_gave_up(ok, fa.fault)) return;  // uniform over the block
  r = group_reduce<OpF, kRowBS>(r);
  if (threadIdx.x == 0) {
    if constexpr (Op::kOrdered) {
      // a NaN at axis position 0 absorbed tile 0 and therefore the whole reduction
      if (first.idx >= 0 && is_nan(first.val)) r = to_final<Op, OpF>(first, 0);
    }
    write_result<OpF, T, kWriteFinal>(out, o, r, 0);
  }
}

// --------------------------------------------------------------------------------------------
// Whole-array reduction (one output): block b of G streams chunks b, b+G, b+2G, ... (chunk =
// one round of the block, kAllBS lanes x UNROLL x 16 bytes; G from launch_reduce_all_fused), folding
// each chunk into its lanes' running accumulators in that fixed order; then blocks publish and a
// combiner block (index G) folds the G block results as in k_reduce_row_fused.  Ordered ops fold
// a chunk with tile-relative int32 indices and move it into an int64 running accumulator per lane.
//
// Walks a block's chunks k = 0 .. mine - 1 through NB register buffers: chunk k lives in buffer
// k % NB, and the loads of chunks k + 1 .. k + NB - 1 are in flight while chunk k is folded.  The
// buffer of every load and fold is a compile-time index (the steady loop is unrolled NB times and
// the last NB - 1 .. 2NB - 2 chunks take one of NB straight-line tails), so no registers are copied
// and no prefetch is conditional: a conditional load would make the wait before each later fold
// cover it too.  `last()` runs once, after the last chunk's loads are issued and before the folds
// that follow them.
template <int NB, class B, class Load, class Fold, class Last>
__device__ inline void walk_chunks(uint64_t mine, B (&buf)[NB], Load&& load, Fold&& fold, Last&& last) {
  static_assert(NB >= 2, "at least two buffers");
  if (mine < uint64_t(NB - 1)) {  // fewer chunks than a full prefetch: all loads, then the folds
    static_for<NB - 1>([&](auto J) { if (J.value < mine) load(uint64_t(J.value), buf[J.value]); });
    last();
    static_for<NB - 1>([&](auto J) { if (J.value < mine) fold(uint64_t(J.value), buf[J.value]); });
    return;
  }
  static_for<NB - 1>([&](auto J) { load(uint64_t(J.value), buf[J.value]); });
  uint64_t k = 0;
  for (; k + 2 * NB - 1 <= mine; k += NB) {
    static_for<NB>([&](auto J) {
      load(k + J.value + NB - 1, buf[(J.value + NB - 1) % NB]);
      fold(k + J.value, buf[J.value]);
    });
  }
  // mine - k = NB - 1 + e chunks are left, 0 <= e < NB; chunks k .. k + NB - 2 are loaded
  const uint32_t e = uint32_t(mine - k) - uint32_t(NB - 1);
  static_for<NB>([&](auto E) {
    if (e == E.value) {
      if constexpr (E.value == 0) last();
      static_for<E.value>([&](auto J) {
        load(k + J.value + NB - 1, buf[(J.value + NB - 1) % NB]);
        if constexpr (J.value + 1 == E.value) last();
        fold(k + J.value, buf[J.value]);
      });
      static_for<NB - 1>([&](auto J) { fold(k + E.value + J.value, buf[(E.value + J.value) % NB]); });
    }
  });
}

// One streaming block's lane accumulator (before the block reduction); `first` receives element 0
// on lane 0 of the block that reads it.
template <class OpF, class T, int VEC, int UNROLL, int BS>
__device__ inline typename OpF::A all_stream(const T* __restrict__ a, uint64_t n, uint32_t grid, uint64_t whole_q,
                                             uint32_t whole_r, uint32_t b, T& first) {
  using AF = typename OpF::A;
  constexpr uint64_t kChunk = uint64_t(BS) * UNROLL * VEC;
  AF acc = OpF::init();
  // The lane's running accumulator (absolute int64 indices) continues from chunk to chunk, so
  // an ordered fold searches a chunk only when the chunk beats it.  Whole chunks are software
  // pipelined: the next kAllBuffers - 1 chunks' loads are in flight while one is folded.
  constexpr uint32_t stepk = uint32_t(BS) * VEC;
  const uint64_t whole = n / kChunk;
  Vec<T, VEC> buf[kAllBuffers][UNROLL];
  // the block's k-th chunk is chunk b + k * grid of the array
  auto load = [&](uint64_t k, Vec<T, VEC>(&dst)[UNROLL]) {
    const T* p = a + (b + k * grid) * kChunk + threadIdx.x * VEC;
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) dst[u] = vload_nt<T, VEC>(p + u * stepk);
  };
  auto fold = [&](uint64_t k, const Vec<T, VEC>(&src)[UNROLL]) {
    const uint64_t cc = b + k * grid;
    T xs[UNROLL][VEC];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int v = 0; v < VEC; ++v) xs[u][v] = src[u].v[v];
    if (cc == 0) first = xs[0][0];  // lane 0 holds element 0
    acc = OpF::template step_chunk<UNROLL, VEC>(acc, xs, threadIdx.x * VEC, stepk, int64_t(cc * kChunk));
  };
  // whole = whole_q * grid + whole_r (from the host: a 64-bit division here would delay every
  // block's first load)
  const uint64_t mine = whole_q + (b < whole_r ? 1 : 0);  // whole chunks of this block
  walk_chunks(mine, buf, load, fold, [] {});
  const uint64_t c = b + mine * grid;  // the first chunk index past this block's whole chunks
  if (c == whole && whole * kChunk < n) {  // the last, partial chunk
    T f{};
    acc = accumulate_segment<OpF, T, BS, VEC, UNROLL>(a + c * kChunk, uint32_t(n - c * kChunk), threadIdx.x, 1,
                                                      f, acc, int64_t(c * kChunk));
    if (c == 0) first = f;
  }
  return acc;
}

template <class Op, class OpF, class T, int VEC, int UNROLL, int PER>
__global__ __launch_bounds__(kAllBS) void k_reduce_all_fused(const T* __restrict__ a, uint64_t n, uint32_t grid,
                                                             uint64_t whole_q, uint32_t whole_r, RedOut<T> out,
                                                             FusedArgs fa) {
  using AF = typename OpF::A;
  static_assert(sizeof(AF) % 4 == 0, "accumulator must split into 32-bit slices");
  constexpr int W = int(sizeof(AF) / 4);
  const uint32_t b = blockIdx.x;
  if (b < grid) {
    T first{};
    AF acc = all_stream<OpF, T, VEC, UNROLL, kAllBS>(a, n, grid, whole_q, whole_r, b, first);
    acc = group_reduce<OpF, kAllBS>(acc, n < 0xffffffffull);
    if (threadIdx.x == 0) {
      if (b == 0 && n > 0) acc = absorb_first<OpF, T>(acc, first);
      uint32_t s[W];
      __builtin_memcpy(s, &acc, sizeof(AF));
      publish_slices<W>(fa.slots + uint64_t(b) * W, s);
    }
    return;
  }
  // combiner: lane l folds block results l, l + kAllBS, ... (PER of them at most)
  uint64_t v[PER][W];
  const bool ok = gather_published<W, PER, kAllBS>(fa.slots, grid, fa.spin_limit, v);
  AF r = OpF::init();
  AF first{};
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t bb = threadIdx.x + j * kAllBS;
    if (bb >= grid) break;
    uint32_t s[W];
#pragma unroll
    for (int i = 0; i < W; ++i) s[i] = uint32_t(v[j][i]);
    AF x;
    __builtin_memcpy(&x, s, sizeof(AF));
    if (bb == 0) first = x;
    r = OpF::comb(r, x);
  }
  if (!combiner_gave_up(ok, fa.fault)) {  // uniform over the block
    r = group_reduce<OpF, kAllBS>(r, n < 0xffffffffull);  // an absorbed NaN is put back below
    if (threadIdx.x == 0) {
      if constexpr (Op::kOrdered) {
        if (first.idx == 0 && is_nan(first.val)) r = first;  // block 0 absorbed a NaN at position 0
      }
      write_result<OpF, T, kWriteFinal>(out, 0, r, 0);
    }
  }
  // The slots go back to zero last: a barrier after these stores would wait for them (on gfx9 a
  // store holds the vector-memory counter that barriers and later loads wait on until it
  // reaches memory), which cost 0.7 us per barrier in the combiner of a 64M argmax.
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t bb = threadIdx.x + j * kAllBS;
    if (bb < grid) {
#pragma unroll
      for (int i = 0; i < W; ++i) st_relaxed(fa.slots + uint64_t(bb) * W + i, 0);
    }
  }
}

// f32 max / min / argmax / argmin over fewer than 2^32 - 1 elements: the same streaming blocks,
// each publishing its result as one key (ext_key_f32, two tagged words), so that the combiner
// folds keys with unsigned maxima.  With the (value, int64 index) accumulator published whole
// (four words), the combiner's gather and fold took 2.8 us after the last block against 0.8 us
// for an f32 sum, and its 8-slot version too many registers for the two-chunk grid.  The NaN at
// position 0 that absorbs the reduction, and the sign of a winning zero, are read back from the
// input by the combiner.
// Keys handed over through one 64-bit word each: the word holds key + 1, so that 0 still means
// "not published" (a key's high word never exceeds 0xff800000, so key + 1 does not wrap) and an
// empty accumulator's key 0 travels as 1.  One word per slot instead of two tagged halves halves
// the combiner's loads and registers: 8 slots per lane at once instead of 4.
__device__ inline void publish_key(uint64_t* slot, uint64_t key) { st_relaxed(slot, key + 1); }

// The largest of `count` published keys (lane l: slots l, l + kRowBS, ...), on thread 0, and
// whether every slot was published within the poll budget (uniform over the block).  The slots go
// back to zero after the block's last barrier, which would otherwise wait for those stores.
template <int PER, int BS = kRowBS>
__device__ inline bool fold_keys(uint64_t* slots, uint64_t count, uint32_t spin_limit, uint32_t* fault,
                                 uint64_t& key) {
  constexpr int kGroup = PER < 8 ? PER : 8;  // slots of a lane gathered at once
  key = 0;
  bool ok = true;
#pragma clang loop unroll(disable)
  for (uint64_t base = 0; base < count; base += uint64_t(kGroup) * BS) {
    uint64_t v[kGroup];
    uint32_t pending = 0;
#pragma unroll
    for (int j = 0; j < kGroup; ++j) {
      v[j] = 0;
      if (base + threadIdx.x + uint64_t(j) * BS < count) pending |= 1u << j;
    }
    for (uint32_t spins = 0; pending != 0 && spins < spin_limit; ++spins) {
#pragma unroll
      for (int j = 0; j < kGroup; ++j)
        if (pending & (1u << j)) v[j] = ld_relaxed(slots + base + threadIdx.x + uint64_t(j) * BS);
#pragma unroll
      for (int j = 0; j < kGroup; ++j)
        if (v[j] != 0) pending &= ~(1u << j);
      if (pending) __builtin_amdgcn_s_sleep(2);
    }
    ok = ok && pending == 0;
#pragma unroll
    for (int j = 0; j < kGroup; ++j) {
      const uint64_t k = v[j] == 0 ? 0 : v[j] - 1;
      key = k > key ? k : key;
    }
  }
  const bool good = !combiner_gave_up(ok, fault);
  if (good) {
#pragma unroll
    for (int m = kWave / 2; m >= 1; m >>= 1) {
      const uint64_t o = acc_shfl(key, m);
      key = o > key ? o : key;
    }
    __shared__ uint64_t part[BS / kWave];
    if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = key;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int i = 1; i < BS / kWave; ++i) key = part[i] > key ? part[i] : key;
    }
  }
  for (uint64_t bb = threadIdx.x; bb < count; bb += BS) st_relaxed(slots + bb, 0);
  return good;
}

template <class Op, class OpF, int UNROLL, int PER>
__global__ __launch_bounds__(kAllBS) void k_reduce_all_keyed(const float* __restrict__ a, uint64_t n, uint32_t grid,
                                                                uint64_t whole_q, uint32_t whole_r, RedOut<float> out,
                                                                FusedArgs fa) {
  using AF = typename OpF::A;
  const uint32_t b = blockIdx.x;
  if (b < grid) {
    float first = 0.0f;
    AF acc = all_stream<OpF, float, 4, UNROLL, kAllBS>(a, n, grid, whole_q, whole_r, b, first);
    acc = group_reduce<OpF, kAllBS>(acc, true);
    if (threadIdx.x == 0) publish_key(fa.slots + b, ext_key_f32<OpF>(acc));
    return;
  }
  const float a0 = a[0];  // loaded while the streaming blocks run
  uint64_t key;
  if (fold_keys<PER, kAllBS>(fa.slots, grid, fa.spin_limit, fa.fault, key) && threadIdx.x == 0) {
    AF r = ext_unkey_f32<OpF, int64_t>(key);
    if (r.idx >= 0 && r.val == 0.0f) r.val = a[r.idx];  // the first zero's own sign
    if (is_nan(a0)) r = AF{a0, 0};  // a NaN at position 0 absorbs the whole reduction
    write_result<OpF, float, kWriteFinal>(out, 0, r, 0);
  }
}

// --------------------------------------------------------------------------------------------
// col kernel: block = (outer, column group, tile); 64 lanes x VEC columns, 4 waves split rows.
struct ColArgs {
  RowIndexer<1> ix;   // outer output dims (all but the innermost one) -> input offset
  uint64_t C;         // innermost output extent (unit stride in the input)
  uint32_t cgroups;   // ceil(C / (64 * VEC))
  uint64_t R;
  int64_t rs;
  uint64_t chunk;
  uint32_t tiles;
};

// A lane's first column.  The last vector of a row of odd length is moved back to end with the row
// (the columns it shares with its neighbour are reduced twice, with the same result).
template <int VEC>
__device__ inline uint64_t lane_col(const ColArgs& ca, uint32_t cg, int lane) {
  const uint64_t c0 = (uint64_t(cg) * kWave + uint64_t(lane)) * VEC;
  return c0 < ca.C && c0 + VEC > ca.C && ca.C >= VEC ? ca.C - VEC : c0;
}

// Sums that round in the element's own type (ordered and integer results are exact, and c64 sums run in
// 64 bits).  The column kernel's 8 waves share the rows of such a sum; a single accumulator for all of
// them measured an error against 64 bits of 3.6e-7 for f32 sums over 572 rows, where that kernel had
// 6.7e-8.  So the lane kernel keeps one accumulator per row in flight and joins them as a tree; the
// span and the column kernel, whose rows are spread over lanes or waves already, add the rows in flight as a
// tree before they meet the accumulator (accumulators of their own would cost the spans the second block
// per CU), and the column kernel's waves meet as a tree: f32 sums over the middle of (64, 2048, 384) 4.6e-8
// against 6.1e-8 with its 4 rows and 8 waves one after the other, 35.7 us both.
template <class Op, class T>
constexpr bool rounds_in_type() {
  return !Op::kOrdered && std::is_same_v<typename Op::A, T>;
}
template <class Op, int N>
__device__ inline typename Op::A tree_fold(typename Op::A (&t)[N]) {
#pragma unroll
  for (int h = N / 2; h > 0; h /= 2)
#pragma unroll
    for (int u = 0; u < h; ++u) t[u] = Op::comb(t[u], t[u + h]);
  return t[0];
}

// One (column group, tile) block of a column reduction: lane `lane` of wave 0 ends with the
// block's accumulators r[v] of its VEC columns (indices relative to the tile) and first[v], the
// elements of axis row 0 when the tile starts there.  `part` is the block's LDS for the waves.
template <class Op, class T, int VEC, int UNROLL, int BS = kRBlock>
__device__ inline void col_partial(const T* __restrict__ a, const ColArgs& ca, uint32_t t, uint32_t cg,
                                   uint32_t outer, typename Op::A (&part)[BS / kWave - 1][kWave * VEC],
                                   typename Op::A (&acc)[VEC], T (&first)[VEC]) {
  using A = typename Op::A;
  constexpr int kWaves = BS / kWave;
  const int lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
  int64_t off[1];
  row_offsets<1>(ca.ix, outer, off);
  const uint64_t c0 = lane_col<VEC>(ca, cg, lane);
  const T* base = a + off[0] + c0;
  const bool full = c0 + VEC <= ca.C;
  const uint64_t k0 = uint64_t(t) * ca.chunk;
  const uint64_t k1 = k0 + ca.chunk < ca.R ? k0 + ca.chunk : ca.R;
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    acc[v] = Op::init();
    first[v] = T{};
  }
  if (c0 < ca.C) {
    uint64_t k = k0 + wv;
    if (full) {
      // the axis's row 0 for the NaN-at-0 rule: one extra load by wave 0 of tile 0, kept out of
      // the streaming loop (a capture inside it cost the ordered kernels ~10% on (8192, 8192))
      if (Op::kOrdered && k == 0 && k < k1) {
        const Vec<T, VEC> x = vload_el<T, VEC>(base);
#pragma unroll
        for (int v = 0; v < VEC; ++v) first[v] = x.v[v];
      }
      // rounds of UNROLL rows (k, k + kWaves, ...).  Ordered ops are software pipelined: the
      // next round's loads are in flight while the current one is folded -- their fold takes
      // its first-index search in most rounds on random data, and with one wave per SIMD nothing
      // else hides it (max over (8192, 8192) axis 0: 50.9 -> 46.2 us).  Sums keep one round in
      // flight (pipelined: 42.9 -> 44.5 us).
      constexpr uint64_t kStep = uint64_t(UNROLL) * kWaves;
      const uint64_t lastu = uint64_t(UNROLL - 1) * kWaves;
      const uint64_t rounds = k + lastu < k1 ? (k1 - k - lastu - 1) / kStep + 1 : 0;
      Vec<T, VEC> x[UNROLL], y[UNROLL];  // ping-pong buffers
      auto load = [&](uint64_t kk, Vec<T, VEC>(&d)[UNROLL]) {
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) d[u] = vload_el<T, VEC>(base + int64_t(kk + u * kWaves) * ca.rs);
      };
      auto fold = [&](uint64_t kk, const Vec<T, VEC>(&src)[UNROLL]) {
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
          T xs[UNROLL][1];
#pragma unroll
          for (int u = 0; u < UNROLL; ++u) xs[u][0] = src[u].v[v];
          if constexpr (rounds_in_type<Op, T>()) {
            A p[UNROLL];
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) p[u] = xs[u][0];
            acc[v] = Op::comb(acc[v], tree_fold<Op>(p));
          } else {
            acc[v] = Op::template step_chunk<UNROLL, 1>(acc[v], xs, uint32_t(kk - k0), uint32_t(kWaves));
          }
        }
      };
      if (!Op::kOrdered) {
        for (uint64_t i = 0; i < rounds; ++i, k += kStep) {
          load(k, x);
          __builtin_amdgcn_sched_barrier(0);
          fold(k, x);
        }
      } else if (rounds > 0) {
        load(k, x);
        uint64_t i = 0;
        for (; i + 2 < rounds; i += 2) {
          load(k + kStep, y);
          fold(k, x);
          load(k + 2 * kStep, x);
          fold(k + kStep, y);
          k += 2 * kStep;
        }
        if (i + 1 < rounds) {
          load(k + kStep, y);
          fold(k, x);
          fold(k + kStep, y);
          k += 2 * kStep;
        } else {
          fold(k, x);
          k += kStep;
        }
      }
      for (; k < k1; k += kWaves) {
        Vec<T, VEC> x = vload_el<T, VEC>(base + int64_t(k) * ca.rs);
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[v] = Op::step(acc[v], x.v[v], int64_t(k - k0));
      }
    } else {
      for (; k < k1; k += kWaves)
#pragma unroll
        for (int v = 0; v < VEC; ++v)
          if (c0 + v < ca.C) {
            const T x = base[int64_t(k) * ca.rs + v];
            if (Op::kOrdered && k == 0) first[v] = x;
            acc[v] = Op::step(acc[v], x, int64_t(k - k0));
          }
    }
  }
  if (wv > 0) {
#pragma unroll
    for (int v = 0; v < VEC; ++v) part[wv - 1][lane * VEC + v] = acc[v];
  }
  __syncthreads();
  if (wv == 0) {
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      if constexpr (rounds_in_type<Op, T>()) {
        A p[kWaves];
        p[0] = acc[v];
#pragma unroll
        for (int i = 1; i < kWaves; ++i) p[i] = part[i - 1][lane * VEC + v];
        acc[v] = tree_fold<Op>(p);
      } else {
#pragma unroll
        for (int i = 0; i < kWaves - 1; ++i) acc[v] = Op::comb(acc[v], part[i][lane * VEC + v]);
      }
    }
  }
}

template <class Op, class T, int VEC, int UNROLL, int WRITE, int BS = kRBlock>
__global__ __launch_bounds__(BS) void k_reduce_col(const T* __restrict__ a, ColArgs ca, RedOut<T> out) {
  using A = typename Op::A;
  __shared__ A part[BS / kWave - 1][kWave * VEC];
  const uint32_t b = blockIdx.x;
  const uint32_t t = b % ca.tiles;
  const uint32_t rest = b / ca.tiles;
  const uint32_t cg = rest % ca.cgroups;
  const uint32_t outer = rest / ca.cgroups;
  A acc[VEC];
  T first[VEC];
  col_partial<Op, T, VEC, UNROLL, BS>(a, ca, t, cg, outer, part, acc, first);
  const int lane = threadIdx.x % kWave;
  const uint64_t c0 = lane_col<VEC>(ca, cg, lane);
  if (threadIdx.x < kWave && c0 < ca.C) {
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      if (c0 + v >= ca.C) break;
      A r = acc[v];
      if (t == 0 && ca.R > 0) r = absorb_first<Op, T>(r, first[v]);  // wave 0 walked row 0
      const uint64_t o = uint64_t(outer) * ca.C + c0 + v;
      write_result<Op, T, WRITE>(out, o * ca.tiles + t, r, int64_t(t) * int64_t(ca.chunk));
    }
  }
}

// --------------------------------------------------------------------------------------------
// span kernel: column reductions of narrow rows.  A block of `bs` lanes reads `lanes` of them
// (lanes * VEC elements, a whole number m of rows) per step, so every lane keeps the same VEC
// columns for the whole walk and loads are contiguous over the block whatever the row length: 37
// columns of f32 take 481 of 512 lanes (13 rows a step), where 64 lanes per row group of the column
// kernel left 54 of 64 idle.  Rows that are not contiguous, or a strip of wider rows, work the same
// as long as the strip holds whole vectors.  Tile t of a slice takes chunks t, t + tiles, ... of
// m * UNROLL rows, so the blocks in flight read neighbouring memory.  The m row residues meet in
// LDS (a tree over rows: fixed order).  With several tiles the block's accumulators go to `part`
// ([slice][tile][column]) and k_span_final folds them.
struct SpanArgs {
  RowIndexer<1> ix;    // outer output dims -> input offset
  uint32_t C;          // innermost output extent (unit stride in the input)
  uint32_t cw;         // columns per strip (== C when one strip)
  uint32_t strips;
  uint32_t m, lanes;   // rows and lanes per step
  uint32_t tiles;
  uint32_t whole;      // whole chunks (m * UNROLL rows) of a slice
  uint64_t R;
  int64_t rs;
  bool flat;           // rows are contiguous (rs == C, one strip): a vector may run into the next row
};

template <class Op, class T, int VEC, int UNROLL, bool FINAL, class S = T, class O = T>
__global__ __launch_bounds__(kSpanBS) void k_reduce_span(const S* __restrict__ a, SpanArgs sa, RedOut<O> out,
                                                         typename Op::A* __restrict__ part) {
  using A = typename Op::A;
  __shared__ A s[kSpanBS * VEC];
  const uint32_t b = blockIdx.x;
  const uint32_t t = b % sa.tiles;
  const uint32_t rest = b / sa.tiles;
  const uint32_t strip = rest % sa.strips;
  const uint32_t outer = rest / sa.strips;
  int64_t off[1];
  row_offsets<1>(sa.ix, outer, off);
  const uint32_t cbase = strip * sa.cw;
  const uint32_t l = threadIdx.x;
  const uint32_t e = l * VEC;           // the lane's first element of a step (row-major over the strip)
  const uint32_t r0 = e / sa.cw, c0 = e - r0 * sa.cw;
  const uint32_t width = sa.cw < sa.C - cbase ? sa.cw : sa.C - cbase;  // columns of this strip
  const bool live = l < sa.lanes && c0 < width;
  const S* p = a + off[0] + cbase;
  // a strip that ends inside a vector: its last vector moves back to end with the row (columns it
  // shares with its neighbour get the same values twice)
  const int32_t shift = !sa.flat && cbase + c0 + VEC > sa.C ? int32_t(cbase + c0 + VEC - sa.C) : 0;
  const uint32_t step_rows = sa.m * UNROLL;
  A acc[VEC];
  uint32_t rv[VEC];                     // row of element v inside a step
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    acc[v] = Op::init();
    rv[v] = sa.flat ? (e + v) / sa.cw : r0;
  }
  if (live) {
    const S* lp = p + int64_t(r0) * sa.rs + int64_t(c0) - shift;
    const S* safe = sa.flat ? p : p + int64_t(c0) - shift;  // row 0 of the lane's columns
    Vec<S, VEC> buf[2][UNROLL];
    auto load = [&](uint64_t k, Vec<S, VEC>(&d)[UNROLL]) {
      const S* q = lp + int64_t((uint64_t(t) + k * sa.tiles) * step_rows) * sa.rs;
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) d[u] = vload_el<S, VEC>(q + int64_t(uint64_t(u) * sa.m) * sa.rs);
      // (the scheduler would move some of these loads below the tree of the round before)
      if constexpr (rounds_in_type<Op, T>()) __builtin_amdgcn_sched_barrier(0);
    };
    auto fold = [&](uint64_t k, const Vec<S, VEC>(&src)[UNROLL]) {
      const uint32_t row = uint32_t((uint64_t(t) + k * sa.tiles) * step_rows);
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        T xs[UNROLL][1];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) xs[u][0] = T(src[u].v[v]);
        if constexpr (rounds_in_type<Op, T>()) {
          A t[UNROLL];
#pragma unroll
          for (int u = 0; u < UNROLL; ++u) t[u] = xs[u][0];
          acc[v] = Op::comb(acc[v], tree_fold<Op>(t));
        } else {
          acc[v] = Op::template step_chunk<UNROLL, 1>(acc[v], xs, row + rv[v], sa.m);
        }
      }
    };
    const uint64_t mine = t < sa.whole ? (sa.whole - t - 1) / sa.tiles + 1 : 0;
    walk_chunks(mine, buf, load, fold, [] {});
    if (t == sa.whole % sa.tiles && uint64_t(sa.whole) * step_rows < sa.R) {
      // The rows past the last whole chunk, in one round of unconditional loads (a lane without a
      // row reads the slice's first one and drops it): with the loads under a condition the
      // compiler waits for each before the next, 8 round trips of about 1 us.
      const uint64_t base = uint64_t(sa.whole) * step_rows;
      Vec<S, VEC> x[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const uint64_t row = base + uint64_t(u) * sa.m;
        const S* q = row + rv[VEC - 1] < sa.R ? lp + int64_t(row) * sa.rs : safe;
        x[u] = vload_el<S, VEC>(q);
      }
      constexpr bool kTree = rounds_in_type<Op, T>();
      A ts[kTree ? VEC : 1][UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const uint64_t row = base + uint64_t(u) * sa.m;
        if constexpr (kTree) {
#pragma unroll
          for (int v = 0; v < VEC; ++v) ts[v][u] = Op::init();
        }
        if (row + rv[VEC - 1] < sa.R) {
#pragma unroll
          for (int v = 0; v < VEC; ++v) {
            if constexpr (kTree) ts[v][u] = T(x[u].v[v]);
            else acc[v] = Op::step(acc[v], T(x[u].v[v]), int64_t(row + rv[v]));
          }
        } else if (row + rv[0] < sa.R) {  // the vector that the end of the slice cuts (flat rows)
          const S* q = lp + int64_t(row) * sa.rs;
#pragma unroll
          for (int v = 0; v < VEC; ++v)
            if (row + rv[v] < sa.R) {
              if constexpr (kTree) ts[v][u] = T(q[v]);
              else acc[v] = Op::step(acc[v], T(q[v]), int64_t(row + rv[v]));
            }
        }
      }
      if constexpr (kTree) {
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[v] = Op::comb(acc[v], tree_fold<Op>(ts[v]));
      }
    }
  }
  // the m x cw accumulators of the block, in row-major order
  if (live) {
#pragma unroll
    for (int v = 0; v < VEC; ++v)
      if (shift <= int32_t(c0) + v || sa.flat) s[int32_t(e) - shift + v] = acc[v];
  }
  __syncthreads();
  for (uint32_t rows = sa.m; rows > 1;) {
    const uint32_t half = (rows + 1) / 2;
    const uint32_t n = (rows - half) * sa.cw;
    for (uint32_t i = l; i < n; i += blockDim.x) s[i] = Op::comb(s[i], s[i + half * sa.cw]);
    __syncthreads();
    rows = half;
  }
  for (uint32_t i = l; i < width; i += blockDim.x) {
    A r = s[i];
    if constexpr (FINAL) {
      if constexpr (Op::kOrdered) r = absorb_first<Op, T>(r, T(p[i]));
      write_result<Op, T, kWriteFinal, O>(out, uint64_t(outer) * sa.C + cbase + i, r, 0);
    } else {
      part[(uint64_t(outer) * sa.tiles + t) * sa.C + cbase + i] = r;
    }
  }
}

// Folds part[slice][tile][column] over the tiles, in order, and returns the words it read to zero
// (the workspace rule).  A block takes `cb` columns of one slice, kSpanBS / cb lanes per column.
template <class Op, class T, class S = T, class O = T>
__global__ __launch_bounds__(kSpanBS) void k_span_final(const S* __restrict__ a, typename Op::A* __restrict__ part,
                                                        RowIndexer<1> ix, uint32_t C, uint32_t tiles, uint32_t cb,
                                                        uint32_t groups, RedOut<O> out) {
  using A = typename Op::A;
  __shared__ A s[kSpanBS];
  const uint32_t outer = blockIdx.x / groups;
  const uint32_t g = blockIdx.x - outer * groups;
  const uint32_t tl = threadIdx.x / cb, c = threadIdx.x - tl * cb;
  const uint32_t rows = kSpanBS / cb;  // lanes per column
  const uint32_t col = g * cb + c;
  const bool live = tl < rows && col < C;
  A* q = part + uint64_t(outer) * tiles * C + col;
  A acc = Op::init();
  if (live) {
    constexpr int U = 8;
    uint32_t t = tl;
    for (; t + (U - 1) * rows < tiles; t += U * rows) {
      A x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) x[u] = q[uint64_t(t + u * rows) * C];
#pragma unroll
      for (int u = 0; u < U; ++u) acc = Op::comb(acc, x[u]);
    }
    for (; t < tiles; t += rows) acc = Op::comb(acc, q[uint64_t(t) * C]);
  }
  if (tl < rows) s[threadIdx.x] = acc;
  T first{};
  if constexpr (Op::kOrdered) {
    if (live && tl == 0) {
      int64_t off[1];
      row_offsets<1>(ix, outer, off);
      first = T(a[off[0] + col]);
    }
  }
  __syncthreads();
  for (uint32_t n = rows; n > 1;) {
    const uint32_t half = (n + 1) / 2;
    if (tl < n - half) s[threadIdx.x] = Op::comb(s[threadIdx.x], s[threadIdx.x + half * cb]);
    __syncthreads();
    n = half;
  }
  if (live && tl == 0) {
    A r = s[c];
    if constexpr (Op::kOrdered) r = absorb_first<Op, T>(r, first);
    write_result<Op, T, kWriteFinal, O>(out, uint64_t(outer) * C + col, r, 0);
  }
  if (live) {
    constexpr int W = int(sizeof(A) / 4);
    for (uint32_t t = tl; t < tiles; t += rows) {
      uint32_t* w = reinterpret_cast<uint32_t*>(q + uint64_t(t) * C);
#pragma unroll
      for (int i = 0; i < W; ++i) w[i] = 0;
    }
  }
}

// lane kernel: column reductions with enough outputs to fill the GPU with one lane per VEC of
// them.  Each lane walks the whole axis, 8 rows of loads in flight; no LDS, no second level.  Ordered and
// integer folds go in the reference's order, sums that round in their type as rounds_in_type says: (100, 256,
// 5120) f32 77 us (6.8 TB/s), its error against 64 bits that of the column kernel.  The last vector of a row is moved back to end with the row: its columns
// are computed twice, with the same result.
template <class Op, class T, int VEC, int UNROLL, class S = T, class O = T>
__global__ __launch_bounds__(kLaneBS) void k_reduce_lane(const S* __restrict__ a, RowIndexer<1> ix, uint32_t C,
                                                         FastDiv vpr, uint64_t R, int64_t rs, uint32_t items,
                                                         RedOut<O> out) {
  using A = typename Op::A;
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= items) return;
  const uint32_t outer = fd_div(vpr, g);
  uint32_t c0 = (g - outer * vpr.d) * VEC;
  if (c0 + VEC > C) c0 = C - VEC;
  int64_t off[1];
  row_offsets<1>(ix, outer, off);
  const S* p = a + off[0] + c0;
  constexpr int kAcc = rounds_in_type<Op, T>() ? UNROLL : 1;
  A acc[kAcc][VEC];
  T first[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
#pragma unroll
    for (int u = 0; u < kAcc; ++u) acc[u][v] = Op::init();
    first[v] = T{};
  }
  if constexpr (Op::kOrdered) {
    const Vec<S, VEC> x = vload_el<S, VEC>(p);
#pragma unroll
    for (int v = 0; v < VEC; ++v) first[v] = T(x.v[v]);
  }
  uint64_t k = 0;
  for (; k + UNROLL <= R; k += UNROLL) {
    Vec<S, VEC> x[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) x[u] = vload_el<S, VEC>(p + int64_t(k + u) * rs);
    if constexpr (rounds_in_type<Op, T>()) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      T xs[UNROLL][1];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) xs[u][0] = T(x[u].v[v]);
      if constexpr (kAcc == 1) {
        acc[0][v] = Op::template step_chunk<UNROLL, 1>(acc[0][v], xs, uint32_t(k), 1);
      } else {
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) acc[u][v] = Op::step(acc[u][v], xs[u][0], 0);
      }
    }
  }
  if (k < R) {  // the rest in one round of loads; rows past the end read the last row, which is dropped
    Vec<S, VEC> x[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) x[u] = vload_el<S, VEC>(p + int64_t(k + u < R ? k + u : R - 1) * rs);
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      if (k + u >= R) break;
#pragma unroll
      for (int v = 0; v < VEC; ++v)
        acc[u % kAcc][v] = Op::step(acc[u % kAcc][v], T(x[u].v[v]), int64_t(k + u));
    }
  }
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    A t[kAcc];
#pragma unroll
    for (int u = 0; u < kAcc; ++u) t[u] = acc[u][v];
    A r = tree_fold<Op>(t);
    if constexpr (Op::kOrdered) r = absorb_first<Op, T>(r, first[v]);
    write_result<Op, T, kWriteFinal, O>(out, uint64_t(outer) * C + c0 + v, r, 0);
  }
}

// --------------------------------------------------------------------------------------------
// Column sums, products and means in one launch: the (column group, tile) blocks of k_reduce_col
// count themselves in their group's counter as they start and publish wave 0's per-column
// accumulators (tagged relaxed words, publish.hpp) as they finish; the block whose increment
// completed the count folds the group's tiles in tile order, writes the outputs and returns the
// slots and the counter to zero.  Nobody waits but that block, the last of its group to start,
// for blocks already running (combiner blocks polling from the start of the launch measured
// slower than partial + final; counting at the end instead of the start cost 0.35 us more).
template <class Op, class T, int VEC, int UNROLL, int BS>
__global__ __launch_bounds__(BS) void k_reduce_col_last(const T* __restrict__ a, ColArgs ca, RedOut<T> out,
                                                        FusedArgs fa, uint32_t* counters) {
  using A = typename Op::A;
  static_assert(!Op::kOrdered && sizeof(A) % 4 == 0, "value folds of 32-bit slices");
  constexpr int W = int(sizeof(A) / 4);
  __shared__ A part[BS / kWave - 1][kWave * VEC];
  __shared__ uint32_t s_last;
  const uint32_t b = blockIdx.x;
  const uint32_t t = b % ca.tiles;
  const uint32_t group = b / ca.tiles;  // outer * cgroups + column group
  const uint32_t cg = group % ca.cgroups;
  const uint32_t outer = group / ca.cgroups;
  // the block counts itself before it streams, so the atomic's round trip overlaps the loads; the
  // last block to start is the one that folds (it waits, boundedly, for slower blocks' slots)
  uint32_t arrived = 0;
  if (threadIdx.x == 0) arrived = atomicAdd(counters + group, 1u);
  A acc[VEC];
  T first[VEC];
  col_partial<Op, T, VEC, UNROLL, BS>(a, ca, t, cg, outer, part, acc, first);
  const int lane = threadIdx.x % kWave;
  const uint64_t c0 = lane_col<VEC>(ca, cg, lane);
  auto slot = [&](uint32_t tt, int v) {
    return fa.slots + ((uint64_t(group) * ca.tiles + tt) * (kWave * VEC) + uint64_t(lane) * VEC + v) * W;
  };
  if (threadIdx.x < kWave) {
#pragma unroll
    for (int v = 0; v < VEC; ++v)
      if (c0 + v < ca.C) {
        uint32_t sl[W];
        __builtin_memcpy(sl, &acc[v], sizeof(A));
        publish_slices<W>(slot(t, v), sl);
      }
  }
  if (threadIdx.x == 0) s_last = arrived == ca.tiles - 1 ? 1u : 0u;
  __syncthreads();
  if (s_last == 0) return;
  // The group's last block.  Each round, wave w reads tile t0 + w (every lane its VEC columns, all
  // words in one round trip) into LDS and clears it; wave 0 then folds the round's tiles in order.
  constexpr int kWaves = BS / kWave;
  __shared__ A g[kWaves][kWave * VEC];
  const int wv = threadIdx.x / kWave;
  A r[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) r[v] = Op::init();
  bool ok = true;
  for (uint32_t t0 = 0; t0 < ca.tiles; t0 += kWaves) {
    const uint32_t tt = t0 + wv;
    if (tt < ca.tiles && c0 < ca.C) {
      uint64_t w[VEC][W];
      uint32_t pending = 0;
#pragma unroll
      for (int v = 0; v < VEC; ++v)
        if (c0 + v < ca.C) pending |= 1u << v;
      for (uint32_t spins = 0; pending != 0 && spins < fa.spin_limit; ++spins) {  // a limit of 0: no poll
#pragma unroll
        for (int v = 0; v < VEC; ++v)
          if (pending & (1u << v))
#pragma unroll
            for (int q = 0; q < W; ++q) w[v][q] = ld_relaxed(slot(tt, v) + q);
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
          bool ready = true;
#pragma unroll
          for (int q = 0; q < W; ++q) ready = ready && (w[v][q] & kTag);
          if (ready) pending &= ~(1u << v);
        }
        if (pending) __builtin_amdgcn_s_sleep(2);
      }
      ok = ok && pending == 0;
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        if (c0 + v >= ca.C) break;
        A x = Op::init();
        if (!(pending & (1u << v))) {
          uint32_t sl[W];
#pragma unroll
          for (int q = 0; q < W; ++q) sl[q] = uint32_t(w[v][q]);
          __builtin_memcpy(&x, sl, sizeof(A));
        }
        g[wv][lane * VEC + v] = x;
#pragma unroll
        for (int q = 0; q < W; ++q) st_relaxed(slot(tt, v) + q, 0);
      }
    }
    __syncthreads();
    if (wv == 0 && c0 < ca.C) {
      for (int k = 0; k < kWaves && t0 + k < ca.tiles; ++k)
#pragma unroll
        for (int v = 0; v < VEC; ++v) r[v] = Op::comb(r[v], g[k][lane * VEC + v]);
    }
    __syncthreads();
  }
  if (__syncthreads_or(ok ? 0 : 1) != 0) {  // a wait ran out: record it and leave the outputs unwritten
    if (threadIdx.x == 0) atomicOr(fa.fault, kFaultReduceWait);
  } else if (wv == 0 && c0 < ca.C) {
#pragma unroll
    for (int v = 0; v < VEC; ++v)
      if (c0 + v < ca.C) write_result<Op, T, kWriteFinal>(out, uint64_t(outer) * ca.C + c0 + v, r[v], 0);
  }
  if (threadIdx.x == 0) __hip_atomic_store(counters + group, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// --------------------------------------------------------------------------------------------
// max / min over both axes of a C-contiguous (R, C) array in one launch, with the result the
// reference's two passes give (reduce_multi, reduction.rs:118-155: axis 0 with keepdims, then
// axis 1).  Pass 1 keeps, per column, the first row holding the column's extreme, and a column
// whose row-0 element is NaN becomes NaN; pass 2 keeps the first column holding the extreme of
// those columns and skips NaN ones, unless column 0 is NaN, which absorbs everything.  So the
// result is the element of extreme value that comes first in COLUMN-major order, among the
// non-NaN elements of the columns whose row-0 element is not NaN -- or x[0][0] when that is NaN.
// The streaming blocks are the column kernel's (column group, row tile) blocks; wave 0 then folds
// its lanes' columns into one (value, col * R + row) key, skipping columns whose row 0 is NaN,
// and publishes it; the last block of the grid combines the published keys in a fixed order.
template <class Op, class OpF, class T, int VEC, int UNROLL, int BS, int PER>
__global__ __launch_bounds__(BS) void k_reduce_col2d(const T* __restrict__ a, ColArgs ca, uint32_t nblk,
                                                     RedOut<T> out, FusedArgs fa) {
  using A = typename Op::A;
  using AF = typename OpF::A;
  static_assert(sizeof(AF) % 4 == 0, "accumulator must split into 32-bit slices");
  constexpr int W = int(sizeof(AF) / 4);
  __shared__ A part[BS / kWave - 1][kWave * VEC];
  const uint32_t b = blockIdx.x;
  const bool idx32 = ca.R * ca.C < 0xffffffffull;
  if (b < nblk) {
    const uint32_t t = b % ca.tiles;
    const uint32_t cg = b / ca.tiles;
    // which of wave 0's columns head with a NaN (pass 2 drops them): read before the stream, so
    // the loads overlap it
    const uint64_t c0 = lane_col<VEC>(ca, cg, threadIdx.x % kWave);
    uint32_t nan_head = 0;
    if (threadIdx.x < kWave) {
#pragma unroll
      for (int v = 0; v < VEC; ++v)
        if (c0 + v < ca.C && is_nan(a[c0 + v])) nan_head |= 1u << v;
    }
    A acc[VEC];
    T first[VEC];
    col_partial<Op, T, VEC, UNROLL, BS>(a, ca, t, cg, 0, part, acc, first);
    if (threadIdx.x < kWave) {  // wave 0 holds the block's per-column results
      AF best = OpF::init();
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        const uint64_t col = c0 + v;
        if (col < ca.C && acc[v].idx >= 0 && !(nan_head & (1u << v)))
          best = OpF::comb(best, AF{acc[v].val, int64_t(col) * int64_t(ca.R) + int64_t(t) * int64_t(ca.chunk) +
                                                    int64_t(acc[v].idx)});
      }
      best = group_reduce<OpF, kWave>(best, idx32);
      if (threadIdx.x == 0) {
        uint32_t s[W];
        __builtin_memcpy(s, &best, sizeof(AF));
        publish_slices<W>(fa.slots + uint64_t(b) * W, s);
      }
    }
    return;
  }
  // combiner: lane l folds keys l, l + BS, ... (PER at most), then the block tree
  uint64_t vv[PER][W];
  const bool ok = gather_published<W, PER, BS>(fa.slots, nblk, fa.spin_limit, vv);
  AF res = OpF::init();
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t bb = threadIdx.x + j * BS;
    if (bb >= nblk) break;
    uint32_t s[W];
#pragma unroll
    for (int i = 0; i < W; ++i) s[i] = uint32_t(vv[j][i]);
    AF xv;
    __builtin_memcpy(&xv, s, sizeof(AF));
    res = OpF::comb(res, xv);
#pragma unroll
    for (int i = 0; i < W; ++i) st_relaxed(fa.slots + uint64_t(bb) * W + i, 0);
  }
  if (combiner_gave_up(ok, fa.fault)) return;  // uniform over the block
  res = group_reduce<OpF, BS>(res, idx32);
  if (threadIdx.x == 0) {
    const T x00 = a[0];
    if (is_nan(x00)) res = AF{x00, 0};  // column 0 is NaN: it absorbs the second pass
    write_result<OpF, T, kWriteFinal>(out, 0, res, 0);
  }
}

// The same two-axis max / min for f32 with rows of at least 2048 elements (16-byte aligned, fewer
// than 2^32 - 1 elements), as row reductions: block r streams row r with the row kernel's access
// pattern and keeps, over the columns whose row-0 element is not NaN (row 0's values are loaded
// beside the row's, from the cache after the first blocks), the extreme and its first column.
// That is the same element: the two-pass result is the column-major first element of extreme value
// among those columns' non-NaN elements, and a row's extreme at its first column, keyed
// (value, column * R + row) (ext_key_f32), is the candidate of that row in column-major order.  Each
// block publishes its key; the last block folds the R keys with unsigned maxima and reads the
// winning zero's sign, and x[0][0] when it is NaN, back from the input.  (8192, 8192): kernel
// 43.7-43.8 us, against 54.2 us for the column-strip kernel (k_reduce_col2d, still used for f64,
// i64 and short rows).  Two rows per block measured slower (52 us: the two rows'
// registers spill at 8 waves per SIMD).
// One lane's extreme over row `row` of C f32 elements (C a multiple of 4), in the row kernel's
// access pattern; with `masked`, elements of columns whose row-0 element (in `a`) is NaN are
// skipped like NaNs.
// With `check` (and not `masked`), row 0's values are loaded beside the row's as well, the fold
// still takes every column, and `nan_seen` tells whether this lane met a NaN in row 0.
template <class Op, int UNROLL>
__device__ inline typename Op::A row_extreme(const float* __restrict__ row, const float* __restrict__ a, uint32_t C,
                                             bool masked, bool check, bool& nan_seen) {
  constexpr int VEC = 4;
  constexpr uint32_t stepk = uint32_t(kRowBS) * VEC;
  const float qn = qnan<float>();
  const bool need_h = masked || check;
  typename Op::A acc = Op::init();
  bool seen = false;
  uint32_t k = uint32_t(threadIdx.x) * VEC;
  for (; k + (UNROLL - 1) * stepk + VEC <= C; k += UNROLL * stepk) {
    Vec<float, VEC> x[UNROLL], h[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) x[u] = vload_nt<float, VEC>(row + k + u * stepk);
    if (need_h) {
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) h[u] = vload<float, VEC>(a + k + u * stepk);
    }
    __builtin_amdgcn_sched_barrier(0);
    float xs[UNROLL][VEC];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        const bool hn = need_h && is_nan(h[u].v[v]);
        seen = seen || hn;
        xs[u][v] = (masked && hn) ? qn : x[u].v[v];
      }
    acc = Op::template step_chunk<UNROLL, VEC>(acc, xs, k, stepk, 0);
  }
  for (; k < C; k += stepk) {  // the rest of the row, in vectors
    const Vec<float, VEC> xv = vload_nt<float, VEC>(row + k);
    Vec<float, VEC> h{};
    if (need_h) h = vload<float, VEC>(a + k);
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      const bool hn = need_h && is_nan(h.v[v]);
      seen = seen || hn;
      acc = Op::step(acc, (masked && hn) ? qn : xv.v[v], int64_t(k + v));
    }
  }
  nan_seen = seen;
  return acc;
}

template <class Op, class OpF, int UNROLL, int PER>
__global__ __launch_bounds__(kRowBS, 8) void k_reduce_rows2d_keyed(const float* __restrict__ a, uint64_t R, uint32_t C,
                                                                   RedOut<float> out, FusedArgs fa) {
  using A = typename Op::A;
  using AF = typename OpF::A;
  const uint64_t b = blockIdx.x;
  // published by block 0: 1 + (row 0 holds a NaN), in kFlagCopies copies 256 bytes apart, so that
  // the polls of the other blocks spread over as many memory channels
  constexpr int kFlagCopies = 64;
  // blocks that check row 0 themselves: one resident generation (256 CUs x 4 blocks of 8 waves)
  constexpr uint64_t kSelfCheckBlocks = 1024;
  uint64_t* const flag = fa.slots;
  uint64_t* const keys = fa.slots + kFlagCopies * 32;  // one key word per row
  if (b < R) {
    const float* row = a + b * uint64_t(C);
    __shared__ uint32_t s_nanhead;
    // Which columns count: only those whose row-0 element is not NaN.  The blocks of the first
    // resident generation load row 0 beside their own row (from the cache after the first blocks)
    // and find out themselves whether it holds a NaN; block 0 publishes that.  Later blocks fold
    // their row over every column and read the word at the end (its load is issued first).  Only
    // when row 0 holds a NaN does a block fold its row again, masking with row 0's values.  At
    // (8192, 8192): the first generation waiting for the word instead cost 0.6 us (44.3-44.5 us
    // against 43.7-43.8 us), two generations checking 44.4 us, every block checking 4 us more,
    // and waiting for the word before folding 2.4 us.
    const bool self = b < kSelfCheckBlocks;
    uint64_t f = 0;
    if (!self && threadIdx.x == 0) f = ld_relaxed(flag + (b % kFlagCopies) * 32);
    bool nan_here = false;
    A acc = row_extreme<Op, UNROLL>(row, a, C, false, self, nan_here);
    if (self) {
      f = __syncthreads_or(nan_here ? 1 : 0) != 0 ? 2 : 1;
      if (b == 0 && threadIdx.x < kFlagCopies) st_relaxed(flag + threadIdx.x * 32, f);
      if (threadIdx.x == 0) s_nanhead = uint32_t(f);
    } else if (threadIdx.x == 0) {
      for (uint32_t spins = 1; f == 0 && spins < fa.spin_limit; ++spins) {
        __builtin_amdgcn_s_sleep(2);
        f = ld_relaxed(flag + (b % kFlagCopies) * 32);
      }
      s_nanhead = uint32_t(f);  // 0 when the wait ran out: the block then masks, which is always right
    }
    acc = group_reduce<Op, kRowBS>(acc);  // the row's extreme; its barrier also hands s_nanhead over
    if (s_nanhead != 1) {  // row 0 holds a NaN (or the wait ran out): fold again over the eligible columns
      __syncthreads();     // thread 0 has read the block reduction's partials
      acc = row_extreme<Op, UNROLL>(row, a, C, true, false, nan_here);
      acc = group_reduce<Op, kRowBS>(acc);  // the row's extreme at its first eligible column
    }
    if (threadIdx.x == 0) {
      const uint64_t key =
          acc.idx < 0 ? 0 : ext_key_f32<OpF>(AF{acc.val, int64_t(acc.idx) * int64_t(R) + int64_t(b)});
      publish_key(keys + b, key);
    }
    return;
  }
  // combiner: the R row keys
  const float a0 = a[0];
  // Block 0's flag copies are read here, early (block 0 published them long before this block
  // started with many rows), and returned to zero below only once seen set: a zero stored without
  // reading the word could land before block 0's flag store (nothing orders that store before
  // block 0's key) and leave the flag set for the next launch on this workspace.
  uint64_t fl = 1;
  if (threadIdx.x < kFlagCopies) fl = ld_relaxed(flag + threadIdx.x * 32);
  uint64_t key;
  if (fold_keys<PER>(keys, R, fa.spin_limit, fa.fault, key) && threadIdx.x == 0) {
    AF r = ext_unkey_f32<OpF, int64_t>(key);
    if (r.idx >= 0 && r.val == 0.0f) {  // the first zero's own sign
      const uint64_t col = uint64_t(r.idx) / R, rw = uint64_t(r.idx) % R;
      r.val = a[rw * uint64_t(C) + col];
    }
    if (is_nan(a0)) r = AF{a0, 0};  // column 0 is NaN: it absorbs the second pass
    write_result<OpF, float, kWriteFinal>(out, 0, r, 0);
  }
  if (threadIdx.x < kFlagCopies) {
    for (uint32_t spins = 1; fl == 0 && spins < fa.spin_limit; ++spins) {
      __builtin_amdgcn_s_sleep(2);
      fl = ld_relaxed(flag + threadIdx.x * 32);
    }
    if (fl == 0) atomicOr(fa.fault, kFaultReduceWait);  // reported: the caller zeroes the workspace again
    st_relaxed(flag + threadIdx.x * 32, 0);
  }
}

// max / min over both axes of a C-contiguous f32 (R, C) array whose rows are whole 32 KB chunks
// (C a multiple of kAllChunk, at most 256 chunks per row), in the whole-array reductions' shape:
// G <= 1024 resident 256-lane blocks, block b taking chunks b, b + G, ... (row-major order, so
// chunk c is row c / cpr), 8 loads in flight per lane, the next chunk's loads issued while one is
// folded, plus a combiner block.  Each lane keeps the best key over its elements (ext_key_f32 of
// (value, column * R + row), so that ties go to the first element in column-major order, which is
// what the reference's axis-0-then-axis-1 passes keep); a chunk is searched for its first extreme
// only when its extreme reaches the lane's best.  Row 0 decides which columns count: the blocks
// that hold its chunks (blocks 0 .. cpr - 1, their first chunk) publish, per wave, whether their
// part held a NaN (in kFlag2Copies copies); every block reads them after its last chunk and, only
// when row 0 holds a NaN, folds its chunks again with those columns masked.
constexpr int kFlag2Copies = 16;
constexpr uint64_t kFlag2Stride = 1024;  // words between copies: up to 256 chunks x 4 waves
constexpr uint64_t kAllChunk = uint64_t(kAllBS) * kAllUnroll * 4;  // f32 elements per chunk

template <class OpF>
__device__ inline uint64_t chunk2d_key(uint64_t best, float (&xs)[kAllUnroll][4], const float* row0,
                                       bool masked, uint32_t col0, uint64_t R, uint32_t r) {
  using Op = OpExt<float, OpF::kMax, false, int32_t>;
  float m = xs[0][0];
  if (masked) {
    // columns whose row-0 element is NaN do not count (row0 holds this chunk's row-0 values)
#pragma unroll
    for (int u = 0; u < kAllUnroll; ++u) {
      const Vec<float, 4> h = vload<float, 4>(row0 + (u * kAllBS + threadIdx.x) * 4);
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (is_nan(h.v[v])) xs[u][v] = qnan<float>();
    }
    m = xs[0][0];
  }
#pragma unroll
  for (int u = 0; u < kAllUnroll; ++u)
#pragma unroll
    for (int v = (u == 0 ? 1 : 0); v < 4; ++v) m = Op::pick(m, xs[u][v]);
  if (is_nan(m)) return best;
  // the best key m could have in this chunk (at its lowest column-major index): when it does not
  // beat the lane's best, no element of the chunk can, and the search is skipped
  const uint64_t top = ext_key_f32<OpF>(VI<float, int64_t>{m, int64_t(col0) * int64_t(R) + r});
  if (top <= best) return best;
  typename Op::A c = Op::template step_chunk<kAllUnroll, 4>(Op::init(), xs, threadIdx.x * 4, kAllBS * 4, 0);
  const uint64_t key =
      ext_key_f32<OpF>(VI<float, int64_t>{c.val, int64_t(col0 + uint32_t(c.idx)) * int64_t(R) + r});
  return key > best ? key : best;
}

template <class OpF, int PER>
__global__ __launch_bounds__(kAllBS) void k_reduce_2d_chunks(const float* __restrict__ a, uint64_t R, uint32_t C,
                                                              uint32_t grid, uint64_t whole_q, uint32_t whole_r,
                                                              RedOut<float> out, FusedArgs fa) {
  using AF = typename OpF::A;
  constexpr uint32_t stepk = uint32_t(kAllBS) * 4;
  const uint32_t cpr = C / uint32_t(kAllChunk);
  const uint64_t nch = R * cpr;
  uint64_t* const flags = fa.slots;  // [copy][chunk of row 0][wave]: 1 + (a NaN in that part)
  uint64_t* const keys = fa.slots + kFlag2Copies * kFlag2Stride;
  const uint32_t b = blockIdx.x;
  const int wv = threadIdx.x / kWave;
  if (b < grid) {
    auto rowcol = [&](uint64_t c, uint32_t& r, uint32_t& col0) {
      const uint32_t cc = uint32_t(c);  // R * C < 2^32
      r = cpr == 1 ? cc : cc / cpr;
      col0 = (cc - r * cpr) * uint32_t(kAllChunk);
    };
    Vec<float, 4> buf[kAllBuffers][kAllUnroll];
    auto load = [&](uint64_t c, Vec<float, 4>(&d)[kAllUnroll]) {
      const float* p = a + c * kAllChunk + threadIdx.x * 4;
#pragma unroll
      for (int u = 0; u < kAllUnroll; ++u) d[u] = vload_nt<float, 4>(p + u * stepk);
    };
    uint64_t best = 0;
    auto fold = [&](uint64_t c, const Vec<float, 4>(&d)[kAllUnroll], bool masked) {
      float xs[kAllUnroll][4];
#pragma unroll
      for (int u = 0; u < kAllUnroll; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) xs[u][v] = d[u].v[v];
      uint32_t r, col0;
      rowcol(c, r, col0);
      if (!masked && c == b && b < cpr) {
        // a part of row 0: publish whether it holds a NaN (per wave, no barrier in the stream)
        bool nan = false;
#pragma unroll
        for (int u = 0; u < kAllUnroll; ++u)
#pragma unroll
          for (int v = 0; v < 4; ++v) nan = nan || is_nan(xs[u][v]);
        const bool any = __ballot(nan) != 0;
        if (threadIdx.x % kWave < kFlag2Copies)
          st_relaxed(flags + (threadIdx.x % kWave) * kFlag2Stride + b * (kAllBS / kWave) + wv, any ? 2 : 1);
      }
      best = chunk2d_key<OpF>(best, xs, a + col0, masked, col0, R, r);
    };
    const uint64_t mine = whole_q + (b < whole_r ? 1 : 0);  // nch = whole_q * grid + whole_r (host)
    // row 0's NaN flags: lane l reads flag l of this block's copy.  The first read is issued with
    // the block's last loads, so that its round trip overlaps the last folds (the flags were
    // published at the blocks' first chunks); a flag not yet set is polled (bounded wait; a wait
    // that runs out counts as a NaN, so the block masks, which is always right).
    const uint32_t nflags = cpr * (kAllBS / kWave);
    const uint64_t* fc = flags + (b % kFlag2Copies) * kFlag2Stride;
    uint64_t f0 = 0;  // flag threadIdx.x (the first of the lane's flags)
    auto read_flag = [&]() {
      if (threadIdx.x < nflags && fa.spin_limit > 0) f0 = ld_relaxed(fc + threadIdx.x);
    };
    // the block's k-th chunk is chunk b + k * grid of the array
    walk_chunks(
        mine, buf, [&](uint64_t k, Vec<float, 4>(&d)[kAllUnroll]) { load(b + k * grid, d); },
        [&](uint64_t k, const Vec<float, 4>(&d)[kAllUnroll]) { fold(b + k * grid, d, false); }, read_flag);
    bool nan0 = false;
    for (uint32_t l = threadIdx.x; l < nflags; l += kAllBS) {
      uint64_t f = l == threadIdx.x ? f0 : (fa.spin_limit > 0 ? ld_relaxed(fc + l) : 0);
      for (uint32_t spins = 1; f == 0 && spins < fa.spin_limit; ++spins) {
        __builtin_amdgcn_s_sleep(2);
        f = ld_relaxed(fc + l);
      }
      nan0 = nan0 || f != 1;
    }
    if (__syncthreads_or(nan0 ? 1 : 0)) {  // row 0 holds a NaN: fold the chunks again, masked
      best = 0;
      for (uint64_t c = b; c < nch; c += grid) {
        load(c, buf[0]);
        fold(c, buf[0], true);
      }
    }
    // block max of the lanes' keys
#pragma unroll
    for (int m = kWave / 2; m >= 1; m >>= 1) {
      const uint64_t o = acc_shfl(best, m);
      best = o > best ? o : best;
    }
    __shared__ uint64_t part[kAllBS / kWave];
    if (threadIdx.x % kWave == 0) part[wv] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int i = 1; i < kAllBS / kWave; ++i) best = part[i] > best ? part[i] : best;
      publish_key(keys + b, best);
    }
    return;
  }
  // combiner
  const float a0 = a[0];
  // Row 0's NaN flags are set at their blocks' first chunks, long before the last key: they are
  // read here, while the streaming blocks run, and returned to zero with plain stores once every
  // block has read them (after the keys), so no read is left after the result write.  A flag is
  // cleared only once seen set: a zero stored unseen could land before the flag store it clears.
  const uint32_t nflags = cpr * (kAllBS / kWave);
  for (uint32_t i = threadIdx.x; i < nflags * kFlag2Copies; i += kAllBS) {
    const uint64_t* p = flags + (i / nflags) * kFlag2Stride + (i % nflags);
    uint64_t f = ld_relaxed(p);
    for (uint32_t spins = 1; f == 0 && spins < fa.spin_limit; ++spins) {
      __builtin_amdgcn_s_sleep(2);
      f = ld_relaxed(p);
    }
    if (f == 0) atomicOr(fa.fault, kFaultReduceWait);  // reported: the caller zeroes the workspace again
  }
  uint64_t key;
  if (fold_keys<PER, kAllBS>(keys, grid, fa.spin_limit, fa.fault, key) && threadIdx.x == 0) {
    AF r = ext_unkey_f32<OpF, int64_t>(key);
    if (r.idx >= 0 && r.val == 0.0f) {  // the first zero's own sign
      const uint64_t col = uint64_t(r.idx) / R, rw = uint64_t(r.idx) % R;
      r.val = a[rw * uint64_t(C) + col];
    }
    if (is_nan(a0)) r = AF{a0, 0};  // column 0 is NaN: it absorbs the second pass
    write_result<OpF, float, kWriteFinal>(out, 0, r, 0);
  }
  for (uint32_t i = threadIdx.x; i < nflags * kFlag2Copies; i += kAllBS)
    st_relaxed(flags + (i / nflags) * kFlag2Stride + (i % nflags), 0);
}

// --------------------------------------------------------------------------------------------
// pair kernel (arg final / mid): rows of (value, index) partials, contiguous [out][n]
template <class Op, class T, int GROUP, int WRITE>
__global__ __launch_bounds__(kRBlock) void k_reduce_pairs(const T* __restrict__ pv, const int64_t* __restrict__ pi,
                                                          uint64_t n, uint64_t chunk, uint32_t tiles, uint64_t nwork,
                                                          RedOut<T> out) {
  using A = typename Op::A;
  const uint64_t w = uint64_t(blockIdx.x) * (kRBlock / GROUP) + threadIdx.x / GROUP;
  const int l = threadIdx.x % GROUP;
  A acc = Op::init();
  uint64_t o = 0, t = 0;
  const bool live = w < nwork;
  if (live) {
    o = w / tiles;
    t = w - o * tiles;
    uint64_t k0 = t * chunk, k1 = k0 + chunk < n ? k0 + chunk : n;
    const T* vrow = pv + o * n;
    const int64_t* irow = pi + o * n;
    // 8 pairs per lane in flight before they are combined (the combine is order-free)
    constexpr int U = 8;
    uint64_t k = k0 + l;
    for (; k + uint64_t(U - 1) * GROUP < k1; k += uint64_t(U) * GROUP) {
      T v[U];
      int64_t ix[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        v[u] = vrow[k + u * GROUP];
        ix[u] = irow[k + u * GROUP];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) acc = Op::step_pair(acc, v[u], ix[u]);
    }
    for (; k < k1; k += GROUP) acc = Op::step_pair(acc, vrow[k], irow[k]);
  }
  acc = group_reduce<Op, GROUP>(acc);
  if (live && (GROUP <= kWave ? l == 0 : threadIdx.x == 0)) {
    if (t == 0 && is_nan(pv[o * n]) && pi[o * n] >= 0) {  // the level below was absorbed by x[0]
      acc.val = pv[o * n];
      acc.idx = pi[o * n];
    }
    write_result<Op, T, WRITE>(out, w, acc);
  }
}

// ============================================================================================
// host side
template <class T> constexpr int rvec() { return sizeof(T) >= 16 ? 1 : int(16 / sizeof(T)); }

inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline RowIndexer<1> out_indexer(const ReducePlan& p, int ndims) {
  // first `ndims` output dims (outermost first) as a row indexer, innermost first
  RowIndexer<1> ix{};
  ix.nd = ndims;
  for (int i = 0; i < ndims; ++i) {
    int d = ndims - 1 - i;
    ix.div[i] = make_fastdiv(uint32_t(p.oshape[d]));
    ix.stride[0][i] = p.ostride[d];
  }
  return ix;
}

template <class Op, class T>
constexpr RedKind red_kind() {
  return Op::kOrdered ? RedKind::kOrdered
         : std::is_same_v<T, c64> || std::is_same_v<T, c128> ? RedKind::kComplexSum : RedKind::kSum;
}

// Recommended tiles per output: enough (output, tile) work items to fill 256 CUs several times
// over while each tile still streams a few tens of KB.
inline size_t tiles_hint(const ReducePlan& p, size_t es, RedKind kind) {
  if (p.R <= 1 || p.out_size == 0) return 1;
  if (p.kind == kColReduce) {
    const ColRoute route = col_route(p, es, kind);
    if (route.kind == ColRoute::kLanes) return 1;
    if (route.kind == ColRoute::kSpans) return route.tiles;
    // column tiles: ~256 long-lived blocks (one per CU, 8 loads of 16 bytes in flight per lane)
    // measured best: (8192, 8192) f32 axis 0 at 6.3 TB/s vs 6.0 with 512 blocks of 4 loads;
    // more concurrent row bands lose to HBM row conflicts (32 bands: 4.7-5.6 TB/s); >= 64 rows
    // per tile
    const int vec = int(16 / es) > 0 ? int(16 / es) : 1;
    uint64_t C = p.oshape[p.ond - 1];
    uint64_t blocks = (p.out_size / C) * ceil_div(C, uint64_t(kWave) * vec);
    const uint64_t want_blocks = 256;
    if (blocks >= want_blocks) return 1;
    uint64_t tiles = ceil_div(want_blocks, blocks);
    uint64_t max_tiles = ceil_div(p.R, 64);
    if (tiles > max_tiles) tiles = max_tiles;
    return size_t(tiles < 1 ? 1 : tiles);
  }
  // row segments: one 512-lane block per (output, tile); below ~8K work items a single pass
  // leaves the GPU idle, so large axes are split into tiles of >= 32 KB (one full round of
  // 16-byte loads of the block kernel); reductions of <= 256 KB are not split at all
  const uint64_t want_items = 8192;
  if (p.out_size >= 2048) return 1;
  if (p.out_size * p.R * es <= (uint64_t(256) << 10)) return 1;
  uint64_t tiles = ceil_div(want_items, p.out_size);
  uint64_t max_tiles = ceil_div(p.R * es, 32768);
  if (tiles > max_tiles) tiles = max_tiles;
  return size_t(tiles < 1 ? 1 : tiles);
}

// --------------------------------------------------------------------------------------------
// Short unit-stride rows (at most 128 vectors), many of them: GROUP lanes per row, U rows per group in flight,
// neighbouring groups on neighbouring rows.  The vector that the end of a row cuts is read from
// where it still fits and its elements that belong to the vector before are skipped, so every load
// is a whole 16 bytes.  Against the group kernels with one row each: (300000, 101) f32 sum 70.4 ->
// 20.9 us (5.8 TB/s), (1000000, 33) 54.2 -> 26.2, (3000000, 8) 124.3 -> 19.4, (1000000, 17) f64 64.2
// -> 30.5; max of (1000000, 33) 76.3 -> 40.9, where the compares of each element begin to bind.
template <class Op, class T, int GROUP, int VEC, int U, class S = T, class O = T>
__global__ __launch_bounds__(kRBlock) void k_reduce_short(const S* __restrict__ a, RowIndexer<1> ix, uint32_t R,
                                                          uint32_t rows, RedOut<O> out) {
  using A = typename Op::A;
  constexpr uint32_t kGroups = kRBlock / GROUP;
  const uint32_t l = threadIdx.x % GROUP;
  const uint32_t row0 = blockIdx.x * (kGroups * U) + threadIdx.x / GROUP;
  const S* p[U];
  A acc[U];
  T first[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t row = row0 + u * kGroups < rows ? row0 + u * kGroups : rows - 1;
    int64_t off[1];
    row_offsets<1>(ix, row, off);
    p[u] = a + off[0];
    acc[u] = Op::init();
    first[u] = T{};
  }
  for (uint32_t k = l * VEC; k < R; k += GROUP * VEC) {
    const uint32_t kk = k + VEC <= R ? k : R - VEC;
    Vec<S, VEC> x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = vload_el<S, VEC>(p[u] + kk);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (Op::kOrdered && k == 0) first[u] = T(x[u].v[0]);
      if constexpr (rounds_in_type<Op, T>()) {  // as a tree, like the lanes after it
        A t[VEC];
#pragma unroll
        for (int v = 0; v < VEC; ++v) t[v] = kk + v >= k ? A(T(x[u].v[v])) : Op::init();
        acc[u] = Op::comb(acc[u], tree_fold<Op>(t));
      } else {
#pragma unroll
        for (int v = 0; v < VEC; ++v)
          if (kk + v >= k) acc[u] = Op::step(acc[u], T(x[u].v[v]), int64_t(kk + v));
      }
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    A r = group_reduce<Op, GROUP>(acc[u]);
    const uint32_t row = row0 + u * kGroups;
    if (l == 0 && row < rows) write_result<Op, T, kWriteFinal, O>(out, row, absorb_first<Op, T>(r, first[u]), 0);
  }
}

// Lanes per row: enough for the row in one step (two from 65 vectors on).  Fewer lanes walking more
// steps each spread a load instruction over more lines: (300000, 101) f32 sum 20.9 us with 32 lanes,
// 28.4 with up to 2 steps, 38.4 with up to 4; (3000000, 8) 19.4 us with 2 lanes, 31.9 with 1.
inline int short_group(uint64_t vecs) {
  int g = 1;
  while (g < kWave && uint64_t(g) < vecs) g *= 2;
  return g;
}
template <class Op, class T, int VEC, class S, class O>
bool launch_short(const S* a, RedOut<O> out, const ReducePlan& p, hipStream_t st) {
  const uint64_t vecs = ceil_div(p.R, uint64_t(VEC));
  if (p.rstride != 1 || p.R < uint64_t(VEC) || vecs > 2 * kWave || p.out_size >= (uint64_t(1) << 31)) return false;
  if (std::is_same_v<S, T> && !short_rows_pay(p.R, vecs, sizeof(typename Op::A), Op::kOrdered)) return false;
  constexpr int U = sizeof(typename Op::A) <= 8 ? 4 : 2;
  const int g = short_group(vecs);
  // below two blocks per CU the rows in flight per group leave the GPU idle: (256, 256) f32 argmax
  // 4.4 us, against 3.7 with a wave per row
  if (ceil_div(p.out_size, uint64_t(kRBlock / g) * U) < 512) return false;
  const RowIndexer<1> ix = out_indexer(p, p.ond);
  const uint32_t R = uint32_t(p.R), rows = uint32_t(p.out_size);
  auto go = [&](auto G) {
    constexpr int kG = decltype(G)::value;
    const unsigned grid = unsigned(ceil_div(rows, uint64_t(kRBlock / kG) * U));
    k_reduce_short<Op, T, kG, VEC, U, S, O><<<grid, kRBlock, 0, st>>>(a, ix, R, rows, out);
  };
  switch (g) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 8: go(std::integral_constant<int, 8>{}); break;
    case 16: go(std::integral_constant<int, 16>{}); break;
    case 32: go(std::integral_constant<int, 32>{}); break;
    default: go(std::integral_constant<int, 64>{}); break;
  }
  return true;
}

// The span route in one launch (one tile) or two (partials in `part`, folded and zeroed by the
// second); `part_bytes` limits the tiles.
template <class Op, class T>
void launch_reduce_span(const T* a, RedOut<T> out, const ReducePlan& p, const ColRoute& r, typename Op::A* part,
                        size_t part_bytes, hipStream_t st) {
  constexpr int V = rvec<T>();
  SpanArgs sa{};
  sa.ix = out_indexer(p, p.ond - 1);
  sa.C = uint32_t(p.oshape[p.ond - 1]);
  sa.cw = r.cw;
  sa.strips = r.strips;
  sa.m = r.m;
  sa.lanes = r.lanes;
  const uint64_t room = part_bytes / (p.out_size * sizeof(typename Op::A));
  sa.tiles = room < r.tiles ? uint32_t(room < 1 ? 1 : room) : r.tiles;
  sa.R = p.R;
  sa.rs = p.rstride;
  sa.whole = uint32_t(p.R / (uint64_t(r.m) * kSpanUnroll));
  sa.flat = r.flat;
  const uint64_t outer = p.out_size / sa.C;
  const dim3 grid(unsigned(outer * sa.strips * sa.tiles));
  if (sa.tiles == 1) {
    k_reduce_span<Op, T, V, kSpanUnroll, true><<<grid, r.bs, 0, st>>>(a, sa, out, part);
    return;
  }
  k_reduce_span<Op, T, V, kSpanUnroll, false><<<grid, r.bs, 0, st>>>(a, sa, out, part);
  const uint32_t cb = sa.C < 32 ? sa.C : 32;
  const uint32_t groups = uint32_t(ceil_div(sa.C, cb));
  k_span_final<Op, T><<<dim3(unsigned(outer * groups)), kSpanBS, 0, st>>>(a, part, sa.ix, sa.C, sa.tiles, cb, groups,
                                                                         out);
}

template <class Op, class T, int WRITE>
void launch_reduce(const T* a, RedOut<T> out, int ndim, const size_t* shape, const ssize_t* strides, int axis,
                   size_t axis_len, size_t out_size, size_t tiles, hipStream_t st) {
  if (out_size == 0) return;  // axis_len == 0 still writes the identity (0 for sums, 1 for products)
  if (!args_ok(ndim, axis)) return;
  if (tiles < 1) tiles = 1;
  ReducePlan p;
  plan_reduce(p, ndim, shape, strides, axis, axis_len, out_size);
  if (ceil_div(p.R, tiles) >= (uint64_t(1) << 31)) {  // tile-relative indices are 32-bit
    g_wrapper_error = 2;
    return;
  }
  // `tiles` is the caller's partial layout: every slot is written, tiles past the end of the
  // axis hold the operation's "empty" value
  constexpr int V = rvec<T>();
  if constexpr (WRITE == kWriteFinal) {
    if (tiles == 1 && p.R > 0) {
      const ColRoute r = col_route(p, sizeof(T), red_kind<Op, T>());
      if (r.kind == ColRoute::kLanes) {
        const uint32_t C = uint32_t(p.oshape[p.ond - 1]);
        const uint32_t vpr = uint32_t(ceil_div(C, V));
        const uint32_t items = uint32_t(p.out_size / C * vpr);
        const uint32_t bs = lane_block(items);
        k_reduce_lane<Op, T, V, kSpanUnroll><<<dim3(unsigned(ceil_div(items, bs))), bs, 0, st>>>(
            a, out_indexer(p, p.ond - 1), C, make_fastdiv(vpr), p.R, p.rstride, items, out);
        return;
      }
      if (r.kind == ColRoute::kSpans) {
        launch_reduce_span<Op, T>(a, out, p, r, nullptr, 0, st);
        return;
      }
    }
  }
  if constexpr (WRITE == kWriteFinal && V > 1) {
    if (tiles == 1 && launch_short<Op, T, V, T, T>(a, out, p, st)) return;
  }
  if (p.kind == kColReduce && p.oshape[p.ond - 1] < (uint64_t(1) << 31)) {
    ColArgs ca{};
    ca.ix = out_indexer(p, p.ond - 1);
    ca.C = p.oshape[p.ond - 1];
    ca.cgroups = uint32_t(ceil_div(ca.C, uint64_t(kWave) * V));
    ca.R = p.R;
    ca.rs = p.rstride;
    ca.chunk = ceil_div(p.R, tiles);
    ca.tiles = uint32_t(tiles);
    const uint64_t blocks = (p.out_size / ca.C) * ca.cgroups * ca.tiles;
    // sums: 8 waves with 4 rows of loads each (42.4-42.7 us for the (8192, 8192) f32 axis-0
    // partial, against 43.4-43.9 with 4 waves x 8 rows); ordered ops keep 4 waves x 8 rows
    // (46.0 us, against 46.9-47.3 with 8 waves): their pipelined fold wants the registers
    if constexpr (Op::kOrdered)
      k_reduce_col<Op, T, V, 8, WRITE, 256><<<dim3(unsigned(blocks)), 256, 0, st>>>(a, ca, out);
    else
      k_reduce_col<Op, T, V, 4, WRITE, 512><<<dim3(unsigned(blocks)), 512, 0, st>>>(a, ca, out);
    return;
  }
  RowArgs ra{};
  ra.ix = out_indexer(p, p.ond);
  ra.R = p.R;
  ra.rs = p.rstride;
  ra.tiles = uint32_t(tiles);
  uint64_t chunk = ceil_div(p.R, tiles);
  const bool vec_ok = p.rstride == 1;  // rows may start at any element (vload_el)
  bool aligned = al16(a);
  for (int d = 0; d < p.ond; ++d)
    if ((uint64_t(p.ostride[d] < 0 ? -p.ostride[d] : p.ostride[d]) * sizeof(T)) % 16) aligned = false;
  ra.nt = true;
  if (vec_ok && V > 1) chunk = ceil_div(chunk, V) * V;
  ra.chunk = chunk;
  ra.nwork = uint64_t(out_size) * tiles;
  const uint64_t seg = chunk < p.R ? chunk : p.R;
  // a 512-lane block per segment from 16 KB on, or a wave for some max / min / arg (see ordered_waves)
  const bool waves = Op::kOrdered && vec_ok && ordered_waves(seg * sizeof(T), ra.nwork);
  if (seg * sizeof(T) >= 16384 && !waves) {
    unsigned grid = unsigned(ra.nwork);
    if (vec_ok && aligned && chunk % (uint64_t(kRowBS) * V * 4) == 0 && p.R % chunk == 0)
      k_reduce_row<Op, T, kRowBS, kRowBS, V, 4, WRITE, T, T, true><<<grid, kRowBS, 0, st>>>(a, ra, out);
    else if (vec_ok)
      k_reduce_row<Op, T, kRowBS, kRowBS, V, 4, WRITE><<<grid, kRowBS, 0, st>>>(a, ra, out);
    else
      k_reduce_row<Op, T, kRowBS, kRowBS, 1, 8, WRITE><<<grid, kRowBS, 0, st>>>(a, ra, out);
  } else if (seg >= 64) {
    unsigned grid = unsigned(ceil_div(ra.nwork, kRBlock / kWave));
    if (waves)
      k_reduce_row<Op, T, kRBlock, kWave, V, 4, WRITE><<<grid, kRBlock, 0, st>>>(a, ra, out);
    else if (vec_ok)
      k_reduce_row<Op, T, kRBlock, kWave, V, 2, WRITE><<<grid, kRBlock, 0, st>>>(a, ra, out);
    else
      k_reduce_row<Op, T, kRBlock, kWave, 1, 4, WRITE><<<grid, kRBlock, 0, st>>>(a, ra, out);
  } else if (seg >= 8 && ra.rs == 1) {
    // short contiguous segments (e.g. the [out][tiles] partials of a final): 16 lanes per
    // output read one coalesced run instead of one lane striding through it
    unsigned grid = unsigned(ceil_div(ra.nwork, kRBlock / 16));
    k_reduce_row<Op, T, kRBlock, 16, 1, 2, WRITE><<<grid, kRBlock, 0, st>>>(a, ra, out);
  } else {
    unsigned grid = unsigned(ceil_div(ra.nwork, kRBlock));
    k_reduce_row<Op, T, kRBlock, 1, 1, 4, WRITE><<<grid, kRBlock, 0, st>>>(a, ra, out);
  }
}

// final over [out_size][num_partials] contiguous partials: the row kernel with unit stride
template <class Op, class T>
void launch_final(const T* partials, RedOut<T> out, size_t num_partials, size_t out_size, hipStream_t st) {
  size_t shape[2] = {out_size, num_partials};
  ssize_t strides[2] = {ssize_t(num_partials), 1};
  launch_reduce<Op, T, kWriteFinal>(partials, out, 2, shape, strides, 1, num_partials, out_size, 1, st);
}

template <class Op, class T, int WRITE>
void launch_pairs(const T* pv, const int64_t* pi, RedOut<T> out, size_t n, size_t out_size, size_t tiles,
                  hipStream_t st) {
  if (out_size == 0 || n == 0) return;
  if (tiles < 1) tiles = 1;
  uint64_t chunk = ceil_div(n, tiles);
  uint64_t nwork = uint64_t(out_size) * tiles;
  if (chunk >= 2048) {  // long segments: a whole block per (output, tile)
    k_reduce_pairs<Op, T, kRBlock, WRITE><<<unsigned(nwork), kRBlock, 0, st>>>(pv, pi, n, chunk, uint32_t(tiles), nwork, out);
  } else {
    unsigned grid = unsigned(ceil_div(nwork, kRBlock / kWave));
    k_reduce_pairs<Op, T, kWave, WRITE><<<grid, kRBlock, 0, st>>>(pv, pi, n, chunk, uint32_t(tiles), nwork, out);
  }
}

// count produced by "+1" repeated axis_len times in T (cpu_mean_typed, op_builder.rs:3608-3612)
template <class T> inline double mean_count(size_t n) {
  if (sizeof(T) == 4) return double(n > (size_t(1) << 24) ? (size_t(1) << 24) : n);
  return double(n > (size_t(1) << 53) ? (size_t(1) << 53) : n);
}

template <class T> inline RedOut<T> vout(T* c) { return RedOut<T>{c, nullptr, 0.0, kFinPlain}; }
template <class T> inline RedOut<T> iout(int64_t* c) { return RedOut<T>{nullptr, c, 0.0, kFinPlain}; }
template <class T> inline RedOut<T> mout(T* c, double cnt) { return RedOut<T>{c, nullptr, cnt, kFinMean}; }

// what a single-launch launcher did
enum : int { kFusedLaunched = 0, kFusedNotCovered = -1, kFusedNoRoom = -2 };

template <class Op, class OpF, class T>
int launch_reduce_all_fused(const T* a, RedOut<T> out, uint64_t n, const WsSplit& w, hipStream_t st);

// Column sums, products and means of `tiles` row tiles in one launch (k_reduce_col_last): the
// slots hold groups x tiles x (64 * VEC) accumulators, then one 32-bit counter per group.
template <class Op, class T>
int launch_reduce_col_last(const T* a, RedOut<T> out, const ReducePlan& p, size_t tiles, const WsSplit& w,
                           hipStream_t st) {
  constexpr int V = rvec<T>();
  constexpr uint64_t W = sizeof(typename Op::A) / 4;
  if (p.oshape[p.ond - 1] >= (uint64_t(1) << 31) || ceil_div(p.R, uint64_t(tiles)) >= (uint64_t(1) << 31))
    return kFusedNotCovered;
  ColArgs ca{};
  ca.ix = out_indexer(p, p.ond - 1);
  ca.C = p.oshape[p.ond - 1];
  ca.cgroups = uint32_t(ceil_div(ca.C, uint64_t(kWave) * V));
  ca.R = p.R;
  ca.rs = p.rstride;
  ca.chunk = ceil_div(p.R, uint64_t(tiles));
  ca.tiles = uint32_t(tiles);
  const uint64_t groups = (p.out_size / ca.C) * ca.cgroups;
  const uint64_t blocks = groups * tiles;
  const uint64_t slot_words = groups * tiles * uint64_t(kWave) * V * W;
  if (blocks >= (uint64_t(1) << 31)) return kFusedNotCovered;
  if ((slot_words + ceil_div(groups, uint64_t(2))) * 8 > w.payload_bytes) return kFusedNoRoom;
  FusedArgs fa{};
  fa.slots = w.payload;
  fa.fault = w.fault;
  fa.spin_limit = wait_spin_limit();
  uint32_t* counters = reinterpret_cast<uint32_t*>(fa.slots + slot_words);
  k_reduce_col_last<Op, T, V, 4, 512><<<dim3(unsigned(blocks)), 512, 0, st>>>(a, ca, out, fa, counters);
  return kFusedLaunched;
}

// The fused single launch for a row-kind reduction split into `tiles` tiles.  kFusedNotCovered
// (nothing launched) when the shape does not take the 512-lane block path, kFusedNoRoom when the
// workspace is too small for its slots.
template <class Op, class OpF, class T>
int launch_reduce_fused(const T* a, RedOut<T> out, int ndim, const size_t* shape, const ssize_t* strides, int axis,
                        size_t axis_len, size_t out_size, size_t tiles, void* ws, size_t ws_bytes, hipStream_t st) {
  WsSplit w;
  if (out_size == 0 || axis_len == 0 || tiles < 2 || !ws_split(ws, ws_bytes, w)) return kFusedNotCovered;
  if (!args_ok(ndim, axis)) return kFusedNotCovered;
  ReducePlan p;
  plan_reduce(p, ndim, shape, strides, axis, axis_len, out_size);
  if (p.kind == kColReduce) {
    const ColRoute r = col_route(p, sizeof(T), red_kind<Op, T>());
    if (r.kind == ColRoute::kLanes) {
      launch_reduce<Op, T, kWriteFinal>(a, out, ndim, shape, strides, axis, axis_len, out_size, 1, st);
      return kFusedLaunched;
    }
    if (r.kind == ColRoute::kSpans) {
      launch_reduce_span<Op, T>(a, out, p, r, reinterpret_cast<typename Op::A*>(w.payload), w.payload_bytes, st);
      return kFusedLaunched;
    }
  }
  if constexpr (!Op::kOrdered) {
    if (p.kind == kColReduce) return launch_reduce_col_last<Op, T>(a, out, p, tiles, w, st);
  }
  if (out_size > kFusedMaxOutputs) return kFusedNotCovered;
  // 2048 tiles measured best for 64M f32 (a combiner lane then folds 4)
  if (tiles > kFusedMaxTiles) tiles = kFusedMaxTiles;
  if (p.kind != kRowReduce || p.rstride != 1) return kFusedNotCovered;
  // one output over one contiguous run: the interleaved-chunk grid of launch_reduce_all_fused
  if (out_size == 1) {
    const int r = launch_reduce_all_fused<Op, OpF, T>(a, out, p.R, w, st);
    if (r != kFusedNotCovered) return r;
  }
  constexpr int V = rvec<T>();
  uint64_t chunk = ceil_div(ceil_div(p.R, tiles), uint64_t(V)) * V;
  if (chunk * sizeof(T) < 16384 || chunk >= (uint64_t(1) << 31)) return kFusedNotCovered;
  if (uint64_t(out_size) * tiles >= (uint64_t(1) << 31)) return kFusedNotCovered;
  const uint64_t W = sizeof(typename Op::A) / 4;
  const uint64_t words = uint64_t(out_size) * tiles * W;
  if (words * 8 > w.payload_bytes) return kFusedNoRoom;
  FusedArgs fa{};
  fa.slots = w.payload;
  fa.fault = w.fault;
  fa.spin_limit = wait_spin_limit();
  RowArgs ra{};
  ra.ix = out_indexer(p, p.ond);
  ra.R = p.R;
  ra.rs = 1;
  ra.tiles = uint32_t(tiles);
  ra.chunk = chunk;
  ra.nwork = uint64_t(out_size) * tiles;
  // streaming blocks first, then one combiner per output
  const dim3 grid(unsigned(ra.nwork + out_size));
  switch (ceil_div(tiles, uint64_t(kRowBS))) {
    case 1: k_reduce_row_fused<Op, OpF, T, V, 4, 1><<<grid, kRowBS, 0, st>>>(a, ra, out, fa); break;
    case 2: k_reduce_row_fused<Op, OpF, T, V, 4, 2><<<grid, kRowBS, 0, st>>>(a, ra, out, fa); break;
    default: k_reduce_row_fused<Op, OpF, T, V, 4, 4><<<grid, kRowBS, 0, st>>>(a, ra, out, fa); break;
  }
  return kFusedLaunched;
}

// Whole-array reduction of `n` contiguous, 16-byte aligned elements: G streaming blocks of kAllBS
// lanes (block b takes chunks b, b + G, ...) plus a combiner block, dispatched after them.  G is
// ceil(chunks / 2), at most 1024: 64M f32 runs one round of resident blocks, 8 chunks each.  The
// sums fit five blocks per CU, so their combiner is resident from the start; the keyed arg kernels
// (four per CU) fill the GPU with the streaming blocks, and their combiner starts when the first
// streaming block ends, long before the last.  The combiner polls every 128 cycles.  With 512-lane blocks of 4
// loads per lane, a one-round grid had measured slower (43.0 us against 40.7 us for two chunks per
// block in 4096 blocks, whose later blocks the dispatcher hands to whichever CUs finish first);
// with 256-lane blocks of 8 loads per lane the one-round grid is the fastest measured (see kAllBS).
constexpr uint64_t kAllMaxBlocks = 1024;  // one round of resident 256-lane blocks
template <class Op, class OpF, class T>
int launch_reduce_all_fused(const T* a, RedOut<T> out, uint64_t n, const WsSplit& w, hipStream_t st) {
  constexpr int V = rvec<T>();
  constexpr uint64_t kChunk = uint64_t(kAllBS) * kAllUnroll * V;
  constexpr uint64_t W = sizeof(typename OpF::A) / 4;
  if (n == 0 || !al16(a)) return kFusedNotCovered;
  const uint64_t nchunks = ceil_div(n, kChunk);
  uint64_t grid = ceil_div(nchunks, uint64_t(2));
  if (grid > kAllMaxBlocks) grid = kAllMaxBlocks;
  if (grid < 2) return kFusedNotCovered;
  if (grid * W * 8 > w.payload_bytes) return kFusedNoRoom;
  FusedArgs fa{};
  fa.slots = w.payload;
  fa.fault = w.fault;
  fa.spin_limit = wait_spin_limit();
  const uint32_t g = uint32_t(grid);
  const dim3 blocks(g + 1);
  const uint64_t q = (n / kChunk) / grid;
  const uint32_t r = uint32_t((n / kChunk) % grid);
  const uint64_t per = ceil_div(grid, uint64_t(kAllBS));  // combiner slots per lane, at most 4
  if constexpr (Op::kOrdered && std::is_same_v<T, float>) {
    if (n < 0xffffffffull) {  // one key per block
      if (per == 1)
        k_reduce_all_keyed<Op, OpF, kAllUnroll, 1><<<blocks, kAllBS, 0, st>>>(a, n, g, q, r, out, fa);
      else if (per == 2)
        k_reduce_all_keyed<Op, OpF, kAllUnroll, 2><<<blocks, kAllBS, 0, st>>>(a, n, g, q, r, out, fa);
      else
        k_reduce_all_keyed<Op, OpF, kAllUnroll, 4><<<blocks, kAllBS, 0, st>>>(a, n, g, q, r, out, fa);
      return kFusedLaunched;
    }
  }
  if (per == 1)
    k_reduce_all_fused<Op, OpF, T, V, kAllUnroll, 1><<<blocks, kAllBS, 0, st>>>(a, n, g, q, r, out, fa);
  else if (per == 2)
    k_reduce_all_fused<Op, OpF, T, V, kAllUnroll, 2><<<blocks, kAllBS, 0, st>>>(a, n, g, q, r, out, fa);
  else
    k_reduce_all_fused<Op, OpF, T, V, kAllUnroll, 4><<<blocks, kAllBS, 0, st>>>(a, n, g, q, r, out, fa);
  return kFusedLaunched;
}


// max / min over both axes of a C-contiguous (R, C) array in one launch: f32 rows of whole 32 KB
// chunks in the whole-array grid (k_reduce_2d_chunks, at most 1024 + 1 blocks), other f32 rows of
// at least 2048 elements as keyed rows (k_reduce_rows2d_keyed, R + 1 blocks), the rest with the
// column kernel's tiling (k_reduce_col2d, about 256 blocks); kFusedNotCovered when the shape fits
// none of them
template <class Op, class OpF, class T>
int launch_reduce_2d_ordered(const T* a, RedOut<T> out, uint64_t R, uint64_t C, void* ws, size_t ws_bytes,
                             hipStream_t st) {
  constexpr int V = rvec<T>();
  constexpr int BS = 256;
  WsSplit w;
  if (R == 0 || C == 0 || !ws_split(ws, ws_bytes, w) || R >= (uint64_t(1) << 31) || R * C >= (uint64_t(1) << 62))
    return kFusedNotCovered;
  if constexpr (std::is_same_v<T, float>) {
    // rows of whole 32 KB chunks: the chunked kernel in one round of resident blocks
    const uint64_t cpr = C / kAllChunk;
    if (C % kAllChunk == 0 && cpr <= 256 && R * C < 0xffffffffull && al16(a) &&
        (kFlag2Copies * kFlag2Stride + kAllMaxBlocks) * 8 <= w.payload_bytes) {
      FusedArgs fk{};
      fk.slots = w.payload;
      fk.fault = w.fault;
      fk.spin_limit = wait_spin_limit();
      const uint64_t nch = R * cpr;
      const uint32_t grid = uint32_t(nch < kAllMaxBlocks ? nch : kAllMaxBlocks);
      const dim3 g(grid + 1);
      const uint64_t per = ceil_div(grid, uint64_t(kAllBS));
      const uint64_t q = nch / grid;
      const uint32_t rr = uint32_t(nch % grid);
      if (per == 1)
        k_reduce_2d_chunks<OpF, 1><<<g, kAllBS, 0, st>>>(a, R, uint32_t(C), grid, q, rr, out, fk);
      else if (per == 2)
        k_reduce_2d_chunks<OpF, 2><<<g, kAllBS, 0, st>>>(a, R, uint32_t(C), grid, q, rr, out, fk);
      else
        k_reduce_2d_chunks<OpF, 4><<<g, kAllBS, 0, st>>>(a, R, uint32_t(C), grid, q, rr, out, fk);
      return kFusedLaunched;
    }
    // rows of at least one block round: the row-keyed kernel
    if (C >= 2048 && C % 4 == 0 && C < (uint64_t(1) << 31) && R * C < 0xffffffffull && al16(a) &&
        (64 * 32 + R) * 8 <= w.payload_bytes) {
      FusedArgs fk{};
      fk.slots = w.payload;
      fk.fault = w.fault;
      fk.spin_limit = wait_spin_limit();
      const dim3 g(unsigned(R + 1));
      using OpR = OpExt<float, Op::kMax, false, int32_t>;
      const uint64_t per = ceil_div(R, uint64_t(kRowBS));
      if (per == 1)
        k_reduce_rows2d_keyed<OpR, OpF, 4, 1><<<g, kRowBS, 0, st>>>(a, R, uint32_t(C), out, fk);
      else if (per == 2)
        k_reduce_rows2d_keyed<OpR, OpF, 4, 2><<<g, kRowBS, 0, st>>>(a, R, uint32_t(C), out, fk);
      else if (per <= 4)
        k_reduce_rows2d_keyed<OpR, OpF, 4, 4><<<g, kRowBS, 0, st>>>(a, R, uint32_t(C), out, fk);
      else
        k_reduce_rows2d_keyed<OpR, OpF, 4, 8><<<g, kRowBS, 0, st>>>(a, R, uint32_t(C), out, fk);
      return kFusedLaunched;
    }
  }
  ColArgs ca{};
  ca.ix.nd = 0;
  ca.C = C;
  ca.cgroups = uint32_t(ceil_div(C, uint64_t(kWave) * V));
  ca.R = R;
  ca.rs = int64_t(C);
  // about 256 long-lived blocks, as the column kernel (128: 67 us, 256: 54 us, 512: 53.5 us,
  // 1024: 61 us for (8192, 8192) f32 max)
  uint64_t tiles = ca.cgroups >= 256 ? 1 : ceil_div(256, ca.cgroups);
  const uint64_t max_tiles = ceil_div(R, 64);
  if (tiles > max_tiles) tiles = max_tiles;
  if (tiles < 1) tiles = 1;
  if (uint64_t(ca.cgroups) * tiles > 4 * BS) return kFusedNotCovered;  // the combiner folds up to 1024 keys
  ca.chunk = ceil_div(R, tiles);
  ca.tiles = uint32_t(tiles);
  const uint32_t nblk = uint32_t(uint64_t(ca.cgroups) * tiles);
  const uint64_t W = sizeof(typename OpF::A) / 4;
  if (uint64_t(nblk) * W * 8 > w.payload_bytes) return kFusedNoRoom;
  FusedArgs fa{};
  fa.slots = w.payload;
  fa.fault = w.fault;
  fa.spin_limit = wait_spin_limit();
  const dim3 g(nblk + 1);
  switch (ceil_div(nblk, uint64_t(BS))) {
    case 1: k_reduce_col2d<Op, OpF, T, V, 8, BS, 1><<<g, BS, 0, st>>>(a, ca, nblk, out, fa); break;
    case 2: k_reduce_col2d<Op, OpF, T, V, 8, BS, 2><<<g, BS, 0, st>>>(a, ca, nblk, out, fa); break;
    default: k_reduce_col2d<Op, OpF, T, V, 8, BS, 4><<<g, BS, 0, st>>>(a, ca, nblk, out, fa); break;
  }
  return kFusedLaunched;
}
}  // namespace mpy
