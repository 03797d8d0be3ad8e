// reduce.hip -- the extern "C" surface of the reductions over floating, complex and int64 arrays:
// the reference's `_v2` entry points (kernels/reduction.mu:1342-2055), the single-launch forms, and
// the library's static scratch and wait faults.  The kernels are in reduce_kernels.hpp.
#include "reduce_kernels.hpp"

#include <mutex>

// =============================================================================================
// extern "C" surface (rust/musapy-ops/src/kernels.rs:139-183, 222-305)
using namespace mpy;

namespace mpy {
template <class T> using OpMax = OpExt<T, true, false>;
template <class T> using OpMin = OpExt<T, false, false>;
template <class T> using OpArgmax = OpExt<T, true, true>;
template <class T> using OpArgmin = OpExt<T, false, true>;
template <class T> using OpArgmax64 = OpExt<T, true, true, int64_t>;  // over (value, absolute index) partials
template <class T> using OpArgmin64 = OpExt<T, false, true, int64_t>;

// --------------------------------------------------------------------------------------------
// Device-resident state of the library: `scratch`, the workspace of the no-alloc single-launch
// reduction (musapy_reduce_fused_noalloc_v1).  Its payload is 1 MiB; the 256 bytes after it hold
// the scratch's fault word (the workspace rule of kcommon.hpp: the last 8-byte word), on a cache
// line of its own.  Each GPU the library runs on holds its own copy until the process ends,
// zero-filled by the code object loader (static storage).  In host code the name is a host-side
// stand-in, not a device address: kernels and copies are only ever given the address that
// hipGetSymbolAddress returns for the current device (DeviceState).
constexpr size_t kScratchPayloadBytes = size_t(1) << 20;  // out_size * tiles * W <= 131072 words
constexpr size_t kScratchBytes = kScratchPayloadBytes + 256;
static __device__ __align__(256) uint64_t scratch[kScratchBytes / 8];

constexpr int kMaxDevices = 64;
struct DeviceState {
  uint64_t* scratch;               // device address of `scratch` on this device
  std::atomic<bool> dirty{false};  // a fault was taken: zero the scratch before its next use
};
std::mutex g_state_mu;
std::atomic<bool> g_state_ready[kMaxDevices];
DeviceState g_state[kMaxDevices];
std::atomic<uint32_t> g_spin_limit{1u << 24};

__global__ void k_zero_words(uint64_t* w, uint64_t n) {
  for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x)
    w[i] = 0;
}
// zeroes `bytes` (a multiple of 8) at `p` with a kernel on `st`
hipError_t zero_on(void* p, size_t bytes, hipStream_t st) {
  const uint64_t n = bytes / 8;
  if (n == 0) return hipSuccess;
  const unsigned g = unsigned(n < 65536 * 256 ? (n + 255) / 256 : 65536);
  k_zero_words<<<dim3(g), 256, 0, st>>>(static_cast<uint64_t*>(p), n);
  return hipGetLastError();
}

// The current device's state, its scratch address resolved once per device with that device
// current; nullptr when a HIP call fails.
DeviceState* device_state() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    (void)hipGetLastError();
    return nullptr;
  }
  if (g_state_ready[dev].load(std::memory_order_acquire)) return &g_state[dev];
  std::lock_guard<std::mutex> lk(g_state_mu);
  if (!g_state_ready[dev].load(std::memory_order_relaxed)) {
    void* s = nullptr;
    if (hipGetSymbolAddress(&s, HIP_SYMBOL(scratch)) != hipSuccess || s == nullptr) {
      (void)hipGetLastError();
      return nullptr;
    }
    g_state[dev].scratch = static_cast<uint64_t*>(s);
    g_state_ready[dev].store(true, std::memory_order_release);
  }
  return &g_state[dev];
}

uint32_t wait_spin_limit() { return g_spin_limit.load(std::memory_order_relaxed); }

// Reads the fault word of the workspace [ws, ws + bytes) after the caller's work on `st`; when it
// is set, zeroes the whole workspace on `st` (a publisher that finished after its combiner gave
// up may have left a tag in it) and waits for that.  Returns the fault bits, or -1.
int take_fault_ws(void* ws, size_t bytes, hipStream_t st) {
  WsSplit w;
  if (!ws_split(ws, bytes, w)) return -1;
  uint32_t v = 0;
  if (hipMemcpyAsync(&v, w.fault, sizeof(v), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess) {
    (void)hipGetLastError();
    return -1;
  }
  if (v == 0) return 0;
  if (zero_on(ws, w.payload_bytes + 8, st) != hipSuccess || hipStreamSynchronize(st) != hipSuccess) {
    (void)hipGetLastError();
    return -1;
  }
  return int(v);
}

// one single-launch reduction: kFusedLaunched, kFusedNotCovered or kFusedNoRoom
inline int fused_dispatch(int op, int dtype, const void* a, void* c, int ndim, const size_t* in_shape,
                          const ssize_t* in_strides, int axis, size_t axis_len, size_t out_size, size_t tiles,
                          void* workspace, size_t workspace_bytes, hipStream_t st) {
#define FUSED_PASS ndim, in_shape, in_strides, axis, axis_len, out_size, tiles, workspace, workspace_bytes, st
#define FUSED_CASE(T)                                                                                              \
  {                                                                                                                \
    const T* x = static_cast<const T*>(a);                                                                         \
    T* cv = static_cast<T*>(c);                                                                                    \
    int64_t* ci = static_cast<int64_t*>(c);                                                                        \
    switch (op) {                                                                                                  \
      case MUSAPY_RED_SUM: return launch_reduce_fused<OpSum<T>, OpSum<T>, T>(x, vout<T>(cv), FUSED_PASS);          \
      case MUSAPY_RED_PROD: return launch_reduce_fused<OpProd<T>, OpProd<T>, T>(x, vout<T>(cv), FUSED_PASS);       \
      case MUSAPY_RED_MAX:                                                                                         \
        return launch_reduce_fused<OpMax<T>, OpExt<T, true, false, int64_t>, T>(x, vout<T>(cv), FUSED_PASS);       \
      case MUSAPY_RED_MIN:                                                                                         \
        return launch_reduce_fused<OpMin<T>, OpExt<T, false, false, int64_t>, T>(x, vout<T>(cv), FUSED_PASS);      \
      case MUSAPY_RED_MEAN:                                                                                        \
        if (sizeof(T) == 8 && T(0.5) == T(0)) return kFusedNotCovered; /* integer means go through f64 */          \
        return launch_reduce_fused<OpSum<T>, OpSum<T>, T>(x, mout<T>(cv, mean_count<T>(axis_len)), FUSED_PASS);    \
      case MUSAPY_RED_ARGMAX: return launch_reduce_fused<OpArgmax<T>, OpArgmax64<T>, T>(x, iout<T>(ci), FUSED_PASS); \
      case MUSAPY_RED_ARGMIN: return launch_reduce_fused<OpArgmin<T>, OpArgmin64<T>, T>(x, iout<T>(ci), FUSED_PASS); \
    }                                                                                                              \
    return kFusedNotCovered;                                                                                       \
  }
  // complex: sum, prod and mean (accumulated in f64 components, narrowed once; the mean divides by
  // the f64 axis length, cpu_reduce_cplx, op_builder.rs:3485-3488)
#define FUSED_CPLX(T)                                                                                              \
  {                                                                                                                \
    const T* x = static_cast<const T*>(a);                                                                         \
    T* cv = static_cast<T*>(c);                                                                                    \
    switch (op) {                                                                                                  \
      case MUSAPY_RED_SUM: return launch_reduce_fused<OpSum<T>, OpSum<T>, T>(x, vout<T>(cv), FUSED_PASS);          \
      case MUSAPY_RED_PROD: return launch_reduce_fused<OpProd<T>, OpProd<T>, T>(x, vout<T>(cv), FUSED_PASS);       \
      case MUSAPY_RED_MEAN:                                                                                        \
        return launch_reduce_fused<OpSum<T>, OpSum<T>, T>(x, mout<T>(cv, double(axis_len)), FUSED_PASS);           \
    }                                                                                                              \
    return kFusedNotCovered;                                                                                       \
  }
  switch (dtype) {
    case MUSAPY_DT_F32: FUSED_CASE(float)
    case MUSAPY_DT_F64: FUSED_CASE(double)
    case MUSAPY_DT_I64: FUSED_CASE(int64_t)
    case MUSAPY_DT_C64: FUSED_CPLX(musapy_c64_t)
    case MUSAPY_DT_C128: FUSED_CPLX(musapy_c128_t)
  }
#undef FUSED_CASE
#undef FUSED_CPLX
#undef FUSED_PASS
  return kFusedNotCovered;
}
}  // namespace mpy

#define RED_ARGS int ndim, const size_t *in_shape, const ssize_t *in_strides, int axis, size_t axis_len, size_t out_size
#define RED_PASS ndim, in_shape, in_strides, axis, axis_len, out_size

extern "C" {

static size_t hint(RedKind kind, RED_ARGS, size_t elem_size) {
  if (out_size == 0 || axis_len == 0 || elem_size == 0) return 1;
  if (ndim < 0 || ndim > kMaxDims || (ndim > 0 && (axis < 0 || axis >= ndim))) return 1;  // the launch reports it
  ReducePlan p;
  plan_reduce(p, RED_PASS);
  return tiles_hint(p, elem_size, kind);
}
size_t musapy_reduce_tiles_hint_v2(int op, int dtype, RED_ARGS) {
  const bool sum = op == MUSAPY_RED_SUM || op == MUSAPY_RED_PROD || op == MUSAPY_RED_MEAN;
  const bool cplx = dtype == MUSAPY_DT_C64 || dtype == MUSAPY_DT_C128;
  const size_t es = dtype == MUSAPY_DT_C128 ? 16 : dtype == MUSAPY_DT_F32 ? 4 : 8;
  return hint(!sum ? RedKind::kOrdered : cplx ? RedKind::kComplexSum : RedKind::kSum, RED_PASS, es);
}
size_t musapy_reduce_tiles_hint(RED_ARGS, size_t elem_size) {
  const size_t sum = hint(RedKind::kSum, RED_PASS, elem_size), ext = hint(RedKind::kOrdered, RED_PASS, elem_size);
  return sum > ext ? sum : ext;
}

// value reductions whose final step is the plain accumulator (sum/prod/max/min, real + complex)
#define MPY_RED_FAMILY(NAME, OP, SN, T)                                                                     \
  void musapy_##NAME##_##SN##_v2(const T* a, T* c, RED_ARGS, hipStream_t st) {                              \
    launch_reduce<OP<T>, T, kWriteFinal>(a, vout<T>(c), RED_PASS, 1, st);                                   \
  }                                                                                                         \
  void musapy_##NAME##_small_axis_##SN##_v2(const T* a, T* c, RED_ARGS, int group_size, hipStream_t st) {   \
    (void)group_size;                                                                                       \
    launch_reduce<OP<T>, T, kWriteFinal>(a, vout<T>(c), RED_PASS, 1, st);                                   \
  }                                                                                                         \
  void musapy_##NAME##_partial_##SN##_v2(const T* a, T* partials, RED_ARGS, size_t tiles_per_output,        \
                                         hipStream_t st) {                                                  \
    launch_reduce<OP<T>, T, kWriteVal>(a, vout<T>(partials), RED_PASS, tiles_per_output, st);               \
  }

#define MPY_RED_FINAL_REAL(NAME, OP, SN, T)                                                                 \
  void musapy_##NAME##_final_##SN##_v2(const T* partials, T* c, size_t num_partials, size_t out_size,       \
                                       hipStream_t st) {                                                    \
    launch_final<OP<T>, T>(partials, vout<T>(c), num_partials, out_size, st);                               \
  }
#define MPY_RED_FINAL_CPLX(NAME, OP, SN, T)                                                                 \
  void musapy_##NAME##_final_##SN##_v2(const T* partials, T* c, size_t num_partials, size_t out_size,       \
                                       size_t axis_len, hipStream_t st) {                                   \
    (void)axis_len;                                                                                         \
    launch_final<OP<T>, T>(partials, vout<T>(c), num_partials, out_size, st);                               \
  }

#define MPY_RED_REAL(SN, T)                  \
  MPY_RED_FAMILY(sum, OpSum, SN, T)          \
  MPY_RED_FAMILY(prod, OpProd, SN, T)        \
  MPY_RED_FAMILY(max, OpMax, SN, T)          \
  MPY_RED_FAMILY(min, OpMin, SN, T)          \
  MPY_RED_FINAL_REAL(sum, OpSum, SN, T)      \
  MPY_RED_FINAL_REAL(prod, OpProd, SN, T)    \
  MPY_RED_FINAL_REAL(max, OpMax, SN, T)      \
  MPY_RED_FINAL_REAL(min, OpMin, SN, T)
MPY_RED_REAL(i64, int64_t)
MPY_RED_REAL(f32, float)
MPY_RED_REAL(f64, double)

#define MPY_RED_CPLX(SN, T)                  \
  MPY_RED_FAMILY(sum, OpSum, SN, T)          \
  MPY_RED_FAMILY(prod, OpProd, SN, T)        \
  MPY_RED_FINAL_CPLX(sum, OpSum, SN, T)      \
  MPY_RED_FINAL_CPLX(prod, OpProd, SN, T)
MPY_RED_CPLX(c64, musapy_c64_t)
MPY_RED_CPLX(c128, musapy_c128_t)

// mean: sum partials, divide in the final step.  Real means divide by the reference's "+1"
// count in T (cpu_mean_typed, op_builder.rs:3608-3612); complex means by the f64 axis length
// (cpu_reduce_cplx, op_builder.rs:3485-3488).
#define MPY_RED_MEAN(SN, T, COUNT)                                                                          \
  void musapy_mean_##SN##_v2(const T* a, T* c, RED_ARGS, hipStream_t st) {                                  \
    launch_reduce<OpSum<T>, T, kWriteFinal>(a, mout<T>(c, COUNT(axis_len)), RED_PASS, 1, st);               \
  }                                                                                                         \
  void musapy_mean_small_axis_##SN##_v2(const T* a, T* c, RED_ARGS, int group_size, hipStream_t st) {       \
    (void)group_size;                                                                                       \
    launch_reduce<OpSum<T>, T, kWriteFinal>(a, mout<T>(c, COUNT(axis_len)), RED_PASS, 1, st);               \
  }                                                                                                         \
  void musapy_mean_partial_##SN##_v2(const T* a, T* partials, RED_ARGS, size_t tiles_per_output,            \
                                     hipStream_t st) {                                                      \
    launch_reduce<OpSum<T>, T, kWriteVal>(a, vout<T>(partials), RED_PASS, tiles_per_output, st);            \
  }                                                                                                         \
  void musapy_mean_final_##SN##_v2(const T* partials, T* c, size_t num_partials, size_t out_size,           \
                                   size_t axis_len, hipStream_t st) {                                       \
    launch_final<OpSum<T>, T>(partials, mout<T>(c, COUNT(axis_len)), num_partials, out_size, st);           \
  }
#define MPY_COUNT_F32(n) mean_count<float>(n)
#define MPY_COUNT_F64(n) mean_count<double>(n)
#define MPY_COUNT_LEN(n) double(n)
MPY_RED_MEAN(f32, float, MPY_COUNT_F32)
MPY_RED_MEAN(f64, double, MPY_COUNT_F64)
MPY_RED_MEAN(c64, musapy_c64_t, MPY_COUNT_LEN)
MPY_RED_MEAN(c128, musapy_c128_t, MPY_COUNT_LEN)

// argmax / argmin
#define MPY_RED_ARG(NAME, OP, SN, T)                                                                        \
  void musapy_##NAME##_##SN##_v2(const T* a, int64_t* c, RED_ARGS, hipStream_t st) {                        \
    launch_reduce<OP<T>, T, kWriteFinal>(a, iout<T>(c), RED_PASS, 1, st);                                   \
  }                                                                                                         \
  void musapy_##NAME##_partial_##SN##_v2(const T* a, T* partials_val, int64_t* partials_idx, RED_ARGS,      \
                                         size_t tiles_per_output, hipStream_t st) {                         \
    RedOut<T> o{partials_val, partials_idx, 0.0, kFinPlain};                                                \
    launch_reduce<OP<T>, T, kWritePair>(a, o, RED_PASS, tiles_per_output, st);                              \
  }                                                                                                         \
  void musapy_##NAME##_final_##SN##_v2(const T* partials_val, const int64_t* partials_idx, int64_t* c,      \
                                       size_t num_partials, size_t out_size, hipStream_t st) {              \
    launch_pairs<OP##64<T>, T, kWriteFinal>(partials_val, partials_idx, iout<T>(c), num_partials, out_size, \
                                            1, st);                                                         \
  }                                                                                                         \
  void musapy_##NAME##_mid_##SN##_v2(const T* partials_val, const int64_t* partials_idx, T* out_val,        \
                                     int64_t* out_idx, size_t out_size, size_t tiles_per_output,            \
                                     size_t axis_len, hipStream_t st) {                                     \
    RedOut<T> o{out_val, out_idx, 0.0, kFinPlain};                                                          \
    launch_pairs<OP##64<T>, T, kWritePair>(partials_val, partials_idx, o, axis_len, out_size,               \
                                           tiles_per_output, st);                                           \
  }
MPY_RED_ARG(argmax, OpArgmax, i64, int64_t)
MPY_RED_ARG(argmax, OpArgmax, f32, float)
MPY_RED_ARG(argmax, OpArgmax, f64, double)
MPY_RED_ARG(argmin, OpArgmin, i64, int64_t)
MPY_RED_ARG(argmin, OpArgmin, f32, float)
MPY_RED_ARG(argmin, OpArgmin, f64, double)

// partial + final in one launch (new; see musapy_kernels.h)
int musapy_reduce_fused_v1(int op, int dtype, const void* a, void* c, int ndim, const size_t* in_shape,
                           const ssize_t* in_strides, int axis, size_t axis_len, size_t out_size, size_t tiles,
                           void* workspace, size_t workspace_bytes, hipStream_t st) {
  const int r = fused_dispatch(op, dtype, a, c, RED_PASS, tiles, workspace, workspace_bytes, st);
  return r == kFusedLaunched ? 0 : -1;
}

// max / min over both axes of a C-contiguous (rows, cols) array in one launch, with the result of
// the reference's two per-axis passes (new; see musapy_kernels.h)
int musapy_reduce_2d_ordered_v1(int op, int dtype, const void* a, void* c, size_t rows, size_t cols,
                                void* workspace, size_t workspace_bytes, hipStream_t st) {
  if (op != MUSAPY_RED_MAX && op != MUSAPY_RED_MIN) return -1;
  const bool mx = op == MUSAPY_RED_MAX;
  int r = kFusedNotCovered;
#define RED2D(T)                                                                                                \
  {                                                                                                             \
    const T* x = static_cast<const T*>(a);                                                                      \
    RedOut<T> o = vout<T>(static_cast<T*>(c));                                                                  \
    r = mx ? launch_reduce_2d_ordered<OpExt<T, true, false>, OpExt<T, true, false, int64_t>, T>(                \
                 x, o, rows, cols, workspace, workspace_bytes, st)                                              \
           : launch_reduce_2d_ordered<OpExt<T, false, false>, OpExt<T, false, false, int64_t>, T>(              \
                 x, o, rows, cols, workspace, workspace_bytes, st);                                             \
  }
  switch (dtype) {
    case MUSAPY_DT_F32: RED2D(float) break;
    case MUSAPY_DT_F64: RED2D(double) break;
    case MUSAPY_DT_I64: RED2D(int64_t) break;
  }
#undef RED2D
  return r == kFusedLaunched ? 0 : -1;
}

// The same single launch with the library's static scratch as its workspace (new; no counterpart
// in kernels.rs): for callers that cannot allocate.  Calls that overlap on one device race.  After
// a fault was taken (musapy_kernels_take_fault) the scratch is zeroed first, on this call's stream.
int musapy_reduce_fused_noalloc_v1(int op, int dtype, const void* a, void* c, int ndim, const size_t* in_shape,
                                   const ssize_t* in_strides, int axis, size_t axis_len, size_t out_size,
                                   size_t tiles, hipStream_t st) {
  DeviceState* ds = device_state();
  if (ds == nullptr) return -1;
  if (ds->dirty.load(std::memory_order_acquire)) {
    if (zero_on(ds->scratch, kScratchBytes, st) != hipSuccess) return -1;
    ds->dirty.store(false, std::memory_order_release);
  }
  const int r = fused_dispatch(op, dtype, a, c, RED_PASS, tiles, ds->scratch, kScratchBytes, st);
  if (r == kFusedNoRoom) {
    g_wrapper_error = 5;
    return -2;
  }
  return r == kFusedLaunched ? 0 : -1;
}

// Returns the fault word of the caller's workspace (kFaultReduceWait | kFaultScanWait), read after
// the caller's work on `st`; a fault zeroes the workspace on `st` before returning.
int musapy_kernels_take_fault_ws(void* workspace, size_t workspace_bytes, hipStream_t st) {
  return take_fault_ws(workspace, workspace_bytes, st);
}

// Returns and clears the fault word of the device's no-alloc scratch, read after the caller has
// synchronized the streams whose no-alloc calls it covers.  The scratch itself is zeroed by the
// next no-alloc call on that device, on that call's stream (a clear issued here would not be
// ordered with another stream's work).
int musapy_kernels_take_fault(int device) {
  int prev = 0;
  if (hipGetDevice(&prev) != hipSuccess) return -1;
  if (device != prev && hipSetDevice(device) != hipSuccess) {
    (void)hipGetLastError();
    return -1;
  }
  int result = 0;
  DeviceState* ds = device_state();
  if (ds == nullptr) {
    result = -1;
  } else if (!ds->dirty.load(std::memory_order_acquire)) {  // dirty: taken already, no call since
    WsSplit w;
    ws_split(ds->scratch, kScratchBytes, w);
    uint32_t v = 0;
    if (hipMemcpy(&v, w.fault, sizeof(v), hipMemcpyDeviceToHost) != hipSuccess) {
      result = -1;
    } else if (v != 0) {
      ds->dirty.store(true, std::memory_order_release);
      result = int(v);
    }
  }
  if (result < 0) (void)hipGetLastError();
  if (device != prev) (void)hipSetDevice(prev);
  return result;
}

// Sets how many polls a bounded device wait makes before it gives up and reports a fault; returns
// the previous limit.  0 makes every wait give up at once (used by tests to force the error path
// while every kernel still exits normally).
uint32_t musapy_kernels_set_spin_limit(uint32_t polls) { return g_spin_limit.exchange(polls); }

}  // extern "C"
