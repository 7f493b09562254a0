// ptk_kernels.hip -- gfx950 (MI355X) kernels of the PrimeTTS conv hot path, and the thin C-ABI
// layer (ptk.h) through which the C host code reaches them.
//
// Wide Conv1d / ConvTranspose1d run as one implicit GEMM on the matrix cores: fp32 products as
// three fp16 ones (v_mfma_f32_32x32x16_f16, fp32 accumulation), or on v_mfma_f32_32x32x2_f32 where
// the operands do not fit fp16's range.  GEMM rows are output channels (convT: phase rows
// r*C4 + co, the reference's packed phase layout), columns are output positions, the reduction
// runs over (tap, input channel).  im2col never exists: each wave stages a window of input columns
// per channel chunk in LDS and reads it K times at the K tap shifts.  The two or four waves of a
// workgroup split the input channels and reduce through LDS in a fixed order (deterministic), then the
// epilogue (bias, LeakyReLU/ReLU/scalar ops, residual / branch-sum tensor adds, division) is
// applied on the accumulator values right before the single store.
#include <hip/hip_runtime.h>

#include <atomic>
#include <mutex>

#include <type_traits>

#include <limits.h>
#include <math.h>
#include <stdint.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "ptk.h"

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------------------ error handling
static thread_local char g_err[512];

static void set_err(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
}

#define HCHK(x)                                                                  \
  do {                                                                           \
    hipError_t e_ = (x);                                                         \
    if (e_ != hipSuccess) {                                                      \
      set_err("%s failed: %s (%s:%d)", #x, hipGetErrorString(e_), __FILE__, __LINE__); \
      return -1;                                                                 \
    }                                                                            \
  } while (0)

extern "C" const char *ptk_last_error(void) { return g_err; }

// ------------------------------------------------------------------------------ static scratch
// Device memory for callers that cannot allocate any (ptd_decode_noalloc): one array per GPU,
// loaded with the code object and held until the process ends.  On the host, `scratch` is only a
// stand-in for the symbol; host code uses the device address hipGetSymbolAddress gives for the
// current device (each GPU has its own copy at its own address), kept per device below.  Every
// user of a GPU shares that GPU's array: work that overlaps in time on one GPU races on it.
static __device__ __align__(256) unsigned char scratch[PTK_STATIC_SCRATCH_BYTES];
#define PTK_SCRATCH_MAX_DEVICES 64
static std::mutex g_scratch_lock;
static void *g_scratch_ptr[PTK_SCRATCH_MAX_DEVICES];
// Users of one GPU's scratch are ordered on that GPU: each waits for the work of the one before
// (an event recorded after it), whatever stream either ran on.  The event is made at set-up with
// the address; g_scratch_use[dev] is held from the wait until the record, so two host threads
// cannot both wait on the same predecessor.
static hipEvent_t g_scratch_done[PTK_SCRATCH_MAX_DEVICES];
static bool g_scratch_recorded[PTK_SCRATCH_MAX_DEVICES];
static std::mutex g_scratch_use[PTK_SCRATCH_MAX_DEVICES];

static int scratch_device(int *dev) {
  HCHK(hipGetDevice(dev));
  if (*dev < 0 || *dev >= PTK_SCRATCH_MAX_DEVICES) {
    set_err("static scratch: device %d out of range", *dev);
    return -1;
  }
  return 0;
}

// resolve (once per device, with that device current) the current device's copy of `scratch`
// and make its ordering event
static int scratch_resolve(void **out) {
  int dev = -1;
  if (scratch_device(&dev)) return -1;
  std::lock_guard<std::mutex> lk(g_scratch_lock);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    HCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) {
      set_err("static scratch: hipGetSymbolAddress gave NULL on device %d", dev);
      return -1;
    }
    if (!g_scratch_done[dev]) HCHK(hipEventCreateWithFlags(&g_scratch_done[dev], hipEventDisableTiming));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

extern "C" int ptk_static_scratch(void **p, size_t *bytes) {
  *p = nullptr;
  *bytes = 0;
  if (scratch_resolve(p)) return -1;
  *bytes = PTK_STATIC_SCRATCH_BYTES;
  return 0;
}

static int stream_capturing(hipStream_t st, bool *on) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  HCHK(hipStreamIsCapturing(st, &cs));
  *on = cs != hipStreamCaptureStatusNone;
  return 0;
}

extern "C" int ptk_scratch_acquire(void *s, int *dev_out) {
  int dev = -1;
  void *p;
  *dev_out = -1;
  if (scratch_resolve(&p) || scratch_device(&dev)) return -1;
  g_scratch_use[dev].lock();
  *dev_out = dev;
  bool cap = false;
  hipError_t e = hipSuccess;
  if (stream_capturing((hipStream_t) s, &cap) == 0) {
    if (!cap && g_scratch_recorded[dev]) e = hipStreamWaitEvent((hipStream_t) s, g_scratch_done[dev], 0);
    if (e == hipSuccess) return 0;
    set_err("hipStreamWaitEvent on the static scratch's event failed: %s", hipGetErrorString(e));
  }
  g_scratch_use[dev].unlock();
  *dev_out = -1;
  return -1;
}

extern "C" int ptk_scratch_release(void *s, int dev, int recorded_work) {
  if (dev < 0 || dev >= PTK_SCRATCH_MAX_DEVICES) return -1;
  bool cap = false;
  int rc = stream_capturing((hipStream_t) s, &cap);
  if (rc == 0 && recorded_work && !cap) {
    const hipError_t e = hipEventRecord(g_scratch_done[dev], (hipStream_t) s);
    if (e == hipSuccess) {
      g_scratch_recorded[dev] = true;
    } else {
      set_err("hipEventRecord on the static scratch's event failed: %s", hipGetErrorString(e));
      rc = -1;
    }
  }
  g_scratch_use[dev].unlock();
  return rc;
}

// ------------------------------------------------------------------------------ runtime wrappers
// Device 0 for the calling thread.  The device count is queried once per process; the current
// device is per-thread HIP state, so every thread that creates a context selects it itself (the
// reference brings contexts up from one thread per stream, concurrently).
extern "C" int ptk_init(void) {
  static std::once_flag once;
  static hipError_t count_err = hipSuccess;
  static int ndev = 0;
  std::call_once(once, [] { count_err = hipGetDeviceCount(&ndev); });
  HCHK(count_err);
  if (ndev < 1) {
    set_err("no HIP device");
    return -1;
  }
  thread_local bool selected = false;
  if (!selected) {
    HCHK(hipSetDevice(0));
    selected = true;
    // PT_V21_SYNC, the reference's scheduling mode for host waits (pt_v21_cuda.cu:758-764): 0 spin,
    // 1 blocking, 2 yield (ROCm treats blocking as yield).  Unset: HIP's own choice.  Set once per
    // process, on the first thread to select the device; on a device already active in this
    // process (another library made it so) HIP refuses the change, which is ignored here as the
    // reference ignores it.
    static std::once_flag sync_once;
    std::call_once(sync_once, [] {
      const char *e = getenv("PT_V21_SYNC");
      if (!e) return;
      const int mode = atoi(e);
      const unsigned fl = mode == 0 ? hipDeviceScheduleSpin
                        : mode == 1 ? hipDeviceScheduleBlockingSync
                        : mode == 2 ? hipDeviceScheduleYield : 0u;
      if (fl && hipSetDeviceFlags(fl) != hipSuccess) (void) hipGetLastError();
    });
    // set-up of the static scratch's address for this device, outside any later stream capture;
    // a failure here is reported by the entry point that needs it (which retries), not by init
    void *p;
    if (scratch_resolve(&p)) g_err[0] = 0;
  }
  return 0;
}
extern "C" int ptk_stream_create(void **s) {
  hipStream_t st;
  HCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  *s = (void *) st;
  return 0;
}
extern "C" int ptk_stream_destroy(void *s) {
  HCHK(hipStreamDestroy((hipStream_t) s));
  return 0;
}
// A bounded single-workgroup kernel of dependent ALU work: no memory reads, no waits, one store
// per lane.  Two launches on one hardware queue run one after the other, on two queues at once,
// which is how the servers time the queue placement of their streams.
// (a device symbol the host could read, so the loop and its store are not removed as dead code)
__device__ float ptk_calib_sink[64];
__global__ void __launch_bounds__(64) calib_kernel(int iters, float seed) {
  float v = seed + (float) threadIdx.x;
  for (int i = 0; i < iters; i++) v = v * 0.999f + 0.5f;
  ptk_calib_sink[threadIdx.x] = v;
}
extern "C" int ptk_calib_launch(int iters, void *s) {
  if (iters < 1 || iters > (1 << 22)) {
    set_err("ptk_calib_launch: %d iterations outside [1, 2^22]", iters);
    return -1;
  }
  hipLaunchKernelGGL(calib_kernel, dim3(1), dim3(64), 0, (hipStream_t) s, iters, 1.0f);
  HCHK(hipGetLastError());
  return 0;
}
extern "C" int ptk_stream_sync(void *s) {
  HCHK(hipStreamSynchronize((hipStream_t) s));
  return 0;
}
extern "C" int ptk_stream_query(void *s) {
  hipError_t e = hipStreamQuery((hipStream_t) s);
  if (e == hipSuccess) return 1;
  if (e == hipErrorNotReady) return 0;
  set_err("hipStreamQuery: %s", hipGetErrorString(e));
  return -1;
}
// Failure injection for tests of the error paths: after `skip` more device allocations succeed,
// the next `n` fail as if the device were out of memory (process-wide; nothing reaches the
// device).  n = 0 switches it off.
static std::mutex g_inject_lock;
static int g_inject_skip, g_inject_fail;
extern "C" void ptk_fail_allocs(int skip, int n) {
  std::lock_guard<std::mutex> lk(g_inject_lock);
  g_inject_skip = skip > 0 ? skip : 0;
  g_inject_fail = n > 0 ? n : 0;
}
static bool inject_alloc_failure() {
  std::lock_guard<std::mutex> lk(g_inject_lock);
  if (g_inject_fail <= 0) return false;
  if (g_inject_skip > 0) {
    g_inject_skip--;
    return false;
  }
  g_inject_fail--;
  return true;
}
extern "C" int ptk_malloc(void **p, size_t bytes) {
  if (inject_alloc_failure()) {
    *p = nullptr;
    set_err("hipMalloc(%zu bytes) failed: injected allocation failure", bytes);
    return -1;
  }
  HCHK(hipMalloc(p, bytes ? bytes : 1));
  return 0;
}
extern "C" int ptk_free(void *p) {
  if (p) HCHK(hipFree(p));
  return 0;
}
extern "C" int ptk_h2d_async(void *dst, const void *src, size_t bytes, void *s) {
  if (bytes) HCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, (hipStream_t) s));
  return 0;
}
extern "C" int ptk_d2h_async(void *dst, const void *src, size_t bytes, void *s) {
  if (bytes) HCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, (hipStream_t) s));
  return 0;
}
extern "C" int ptk_d2d_async(void *dst, const void *src, size_t bytes, void *s) {
  if (bytes) HCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, (hipStream_t) s));
  return 0;
}
extern "C" int ptk_fill_async(void *dst, int byte, size_t bytes, void *s) {
  HCHK(hipMemsetAsync(dst, byte, bytes, (hipStream_t) s));
  return 0;
}
extern "C" int ptk_d2d_2d_async(void *dst, size_t dpitch, const void *src, size_t spitch,
                                size_t wb, size_t h, void *s) {
  if (wb && h)
    HCHK(hipMemcpy2DAsync(dst, dpitch, src, spitch, wb, h, hipMemcpyDeviceToDevice, (hipStream_t) s));
  return 0;
}
extern "C" int ptk_d2h_2d_async(void *dst, size_t dpitch, const void *src, size_t spitch,
                                size_t wb, size_t h, void *s) {
  if (wb && h)
    HCHK(hipMemcpy2DAsync(dst, dpitch, src, spitch, wb, h, hipMemcpyDeviceToHost, (hipStream_t) s));
  return 0;
}
extern "C" int ptk_h2d_2d_async(void *dst, size_t dpitch, const void *src, size_t spitch,
                                size_t wb, size_t h, void *s) {
  if (wb && h)
    HCHK(hipMemcpy2DAsync(dst, dpitch, src, spitch, wb, h, hipMemcpyHostToDevice, (hipStream_t) s));
  return 0;
}
extern "C" int ptk_event_create(void **e) {
  hipEvent_t ev;
  HCHK(hipEventCreate(&ev));
  *e = (void *) ev;
  return 0;
}
extern "C" int ptk_event_destroy(void *e) {
  HCHK(hipEventDestroy((hipEvent_t) e));
  return 0;
}
extern "C" int ptk_event_record(void *e, void *s) {
  HCHK(hipEventRecord((hipEvent_t) e, (hipStream_t) s));
  return 0;
}
extern "C" int ptk_stream_wait_event(void *s, void *e) {
  HCHK(hipStreamWaitEvent((hipStream_t) s, (hipEvent_t) e, 0));
  return 0;
}
extern "C" int ptk_event_elapsed_ms(float *ms, void *e0, void *e1) {
  HCHK(hipEventElapsedTime(ms, (hipEvent_t) e0, (hipEvent_t) e1));
  return 0;
}
extern "C" int ptk_event_sync(void *e) {
  HCHK(hipEventSynchronize((hipEvent_t) e));
  return 0;
}
extern "C" int ptk_device_sync(void) {
  HCHK(hipDeviceSynchronize());
  return 0;
}
extern "C" int ptk_capture_begin(void *s) {
  HCHK(hipStreamBeginCapture((hipStream_t) s, hipStreamCaptureModeThreadLocal));
  return 0;
}
extern "C" int ptk_capture_end(void *s, void **exec) {
  hipGraph_t g = nullptr;
  HCHK(hipStreamEndCapture((hipStream_t) s, &g));
  if (!exec) {
    if (g) (void) hipGraphDestroy(g);
    return 0;
  }
  hipGraphExec_t e = nullptr;
  const hipError_t err = hipGraphInstantiate(&e, g, nullptr, nullptr, 0);
  (void) hipGraphDestroy(g);
  HCHK(err);
  *exec = (void *) e;
  return 0;
}
extern "C" int ptk_graph_launch(void *exec, void *s) {
  HCHK(hipGraphLaunch((hipGraphExec_t) exec, (hipStream_t) s));
  return 0;
}
extern "C" int ptk_graph_destroy(void *exec) {
  if (exec) HCHK(hipGraphExecDestroy((hipGraphExec_t) exec));
  return 0;
}

// ------------------------------------------------------------------------------ weight relayout
// The conv kernel multiplies fp32 operands on the fp16 matrix cores: an operand v, scaled by a
// power of two into fp16's range, is taken as two fp16 parts
//     hi = fp16(v),  lo = fp16(v - hi),
// each rounded to nearest even (v - hi is exact in fp32).  Together they hold 23 bits: hi + lo is
// within 2^-23 of v while lo stays a normal fp16, and within half its smallest step below that.
//   Weights are scaled row by row so that the row's largest magnitude lies in [2^14, 2^15): those
//     below 2^-2 (2^-16 of the row's largest) are held to 2^-25 absolute.
//   Inputs take the fixed scale 2^CONV_XS (up to 2^(16 - CONV_XS) fits), and their lo is stored times
//     2^11, which puts its smallest step at 2^-35: inputs are held to 2^-36 absolute.
// A product w x is summed as wl.xh + wh.xh + (wh 2^-11).(xl 2^11), the shifted wh formed in registers.
// Dropping wl.xl costs up to 2^-22 of the product, so that one is within 2^-21 of w x (fp32: 2^-24),
// plus the absolute parts: |w| 2^-35 from the input's side, |x| 2^-24 for a weight below 2^-2.
// Whether those are small beside the products of an output is decided by conv_mfma_kernel with a
// threshold per row that relayout_kernel makes.
//
// Packed [M/4][K][cin][4] (the reference's conv layout; a convT's phase rows are just more rows)
// -> these parts, one after the other (Mp: M rounded up to 32, cinp: cin rounded up to 16; padding
// rows and channels are zero):
//   fp16 [Mp/32][cinp/16][K][2][64][8]: for a row block mb, a chunk of 16 input channels and a tap k,
//     lane l = 32*h + r of a wave holds, of hi and of lo, the eight scaled values
//     W[mb*32 + r][k][chunk*16 + 8*h + e], e = 0..7: its A operand of one v_mfma_f32_32x32x16_f16.
//     One 16-byte load per lane and part; the 2 KiB a wave loads for one (chunk, tap) are
//     contiguous and so are the taps of its chunks.
//   fp32 [Mp/32][cinp/16][K][64][8]: the weights themselves in the same order (conv_mfma_kernel's
//     second pass).
//   fp32 [2][Mp]: per row, the factor 2^-(row exponent + CONV_XS) that takes a sum of products of
//     scaled operands back, and the threshold of that sum (see conv_mfma_kernel).  NaN and inf for a
//     row that has no fp16 form (an inf or NaN weight, or all of it below 2^-100).
//   fp32 [Mp/32]: the largest threshold of each row block.
#define CONV_CK 16         // input channels per staged chunk (per wave)
#define CONV_TAPB 2048     // bytes of one (row block, chunk, tap) of either copy of the weights
// Waves per SIMD the registers are budgeted for, and (chunk, tap) slices the A operands are loaded
// ahead, by column blocks per wave.  A launch small enough for one column block (choose_tiles) has
// about one wave per SIMD and waits for its loads, so it runs further ahead instead.
#ifndef CONV_WPE1
#define CONV_WPE1 3
#define CONV_PD1 4
#define CONV_WPE2 3
#define CONV_PD2 3
#define CONV_LA1 2
#define CONV_LA2 2
#endif
// The inputs' scale, 2^CONV_XS: up to 2^12 an input fits its fp16 parts, and outputs of N(0, s) inputs
// keep to the first pass down to about s = 2^-6, below that all but a few workgroups do (a larger scale
// moves both ends down).
#define CONV_XS 4
#define CONV_LS 2048.0f    // the scale of the inputs' lo

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

extern "C" int ptk_conv_cinp(int cin) { return (cin + CONV_CK - 1) / CONV_CK * CONV_CK; }
extern "C" size_t ptk_relayout_floats(int M, int K, int cin) {
  const size_t Mp = (size_t) (M + 31) / 32 * 32;
  return Mp * (size_t) K * (size_t) ptk_conv_cinp(cin) * 2 + 2 * Mp + Mp / 32;
}

// two floats -> their fp16s (round to nearest even) in one word, a in the low half
__device__ __forceinline__ unsigned f16_pair(float a, float b) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, h2{(_Float16) a, (_Float16) b});
}
// the two parts of a pair of scaled weights
__device__ __forceinline__ void split_pair(float a, float b, unsigned &h, unsigned &l) {
  const _Float16 ha = (_Float16) a, hb = (_Float16) b;
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  h = __builtin_bit_cast(unsigned, h2{ha, hb});
  l = f16_pair(__builtin_fmaf((float) ha, -1.0f, a), __builtin_fmaf((float) hb, -1.0f, b));
}
// and of a pair of inputs, which it scales by 2^CONV_XS (exact: powers of two, and the fma's result is);
// written so that each part is one mixed-precision fma of the input times both scales
__device__ __forceinline__ void split_input(float a, float b, unsigned &h, unsigned &l) {
  const float a2 = a * ((float) (1 << CONV_XS) * CONV_LS), b2 = b * ((float) (1 << CONV_XS) * CONV_LS);
  const _Float16 ha = (_Float16) __builtin_fmaf(a2, 1.0f / CONV_LS, 0.0f), hb = (_Float16) __builtin_fmaf(b2, 1.0f / CONV_LS, 0.0f);
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  h = __builtin_bit_cast(unsigned, h2{ha, hb});
  l = f16_pair(__builtin_fmaf((float) ha, -CONV_LS, a2), __builtin_fmaf((float) hb, -CONV_LS, b2));
}

// Split planes: an activation tensor [C][T] already in two parts, scaled by 2^CONV_XS, as
// [C/8][2][T][8] fp16: per group of eight channels the hi row and the lo row, a column's eight
// channels in 16 bytes.  A conv reads it by copying 16-byte columns into its window, without the
// conversions every row block would repeat.  Same bytes as the fp32 tensor.
//
// il: 0, or the rows per phase C4 (a multiple of 8) of a stride-4 convT whose rows the MFMA layout
// interleaves by phase: a 32-row block holds eight channels, relaid row m is phase (m >> 3) & 3 of
// channel (m >> 5) * 8 + (m & 7), packed row phase * il + channel.
//
// One workgroup per four packed rows, which are contiguous: their largest magnitudes first, then
// (from cache) thread by thread eight channels of one (tap, chunk half) of the four rows.
#define RELAY_THREADS 256
__global__ void __launch_bounds__(RELAY_THREADS) relayout_kernel(
    float *__restrict__ dst, const float *__restrict__ wp, int M, int K, int cin, int cinp, int il) {
  __shared__ unsigned smax[4], snum[4];
  __shared__ unsigned long long sthr[4];
  const int Mp = (M + 31) / 32 * 32, nchunk = cinp / CONV_CK;
  const int tid = threadIdx.x, m0 = blockIdx.x * 4;
  const float4 *src = reinterpret_cast<const float4 *>(wp) + (long long) blockIdx.x * K * cin;
  if (tid < 4) smax[tid] = snum[tid] = 0, sthr[tid] = 0;
  __syncthreads();
  if (m0 < M) {
    unsigned mx[4] = {0, 0, 0, 0};   // as bit patterns: inf and NaN sort above every finite value
    for (int i = tid; i < K * cin; i += RELAY_THREADS) {
      const float4 v = src[i];
      mx[0] = max(mx[0], __float_as_uint(v.x) & 0x7fffffffu);
      mx[1] = max(mx[1], __float_as_uint(v.y) & 0x7fffffffu);
      mx[2] = max(mx[2], __float_as_uint(v.z) & 0x7fffffffu);
      mx[3] = max(mx[3], __float_as_uint(v.w) & 0x7fffffffu);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) atomicMax(&smax[r], mx[r]);
  }
  __syncthreads();
  float up[4], fac[4];
  int row[4];   // relaid rows
  const long long wn = (long long) Mp * K * cinp;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int ms = m0 + r;
    const int c = il ? ms % il : 0;
    row[r] = il && ms < M ? (c >> 3) * 32 + ms / il * 8 + (c & 7) : ms;
    const unsigned mx = smax[r];
    const int e = (int) (mx >> 23) - 127;   // exponent of the largest magnitude
    const bool none = mx == 0, bad = !none && (e < -100 || mx >= 0x7f800000u);
    const int s = none || bad ? 0 : 14 - e;
    up[r] = __uint_as_float((unsigned) (127 + s) << 23);
    fac[r] = bad ? __uint_as_float(0x7fc00000u) : __uint_as_float((unsigned) (127 - s - CONV_XS) << 23);
    if (tid == 0) dst[2 * wn + row[r]] = fac[r];
  }
  // Of each row: the sum of its weights' magnitudes, each rounded up, plus 2^27 for every one below
  // 2^-2 (integers: the same in any order), and the number of nonzero ones.
  unsigned long long ta[4] = {0, 0, 0, 0};
  unsigned nz[4] = {0, 0, 0, 0};
  for (int i = tid; i < nchunk * K * 2; i += RELAY_THREADS) {
    const int h = i & 1, k = (i >> 1) % K, chunk = (i >> 1) / K;
    float v[4][8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int ci = chunk * CONV_CK + 8 * h + e;
      const float4 f = m0 < M && ci < cin ? src[(long long) k * cin + ci] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      v[0][e] = f.x;
      v[1][e] = f.y;
      v[2][e] = f.z;
      v[3][e] = f.w;
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const long long slice = ((long long) (row[r] >> 5) * nchunk + chunk) * K + k;
      const int lane = 32 * h + (row[r] & 31);
      u32x4 hi, lo;
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float m = fabsf(v[r][e] * up[r]);
        if (m > 0.0f && m <= 32768.0f) {
          nz[r]++;
          ta[r] += (unsigned long long) (unsigned) ceilf(m) + (m < 0.25f ? 1ull << 27 : 0ull);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; e++) {
        unsigned a, b;
        split_pair(v[r][2 * e] * up[r], v[r][2 * e + 1] * up[r], a, b);
        hi[e] = a;
        lo[e] = b;
      }
      u32x4 *d16 = reinterpret_cast<u32x4 *>(dst) + slice * (CONV_TAPB / 16) + lane;
      d16[0] = hi;
      d16[64] = lo;
      float4 *d32 = reinterpret_cast<float4 *>(dst + wn) + slice * (CONV_TAPB / 16) + lane * 2;
      d32[0] = make_float4(v[r][0], v[r][1], v[r][2], v[r][3]);
      d32[1] = make_float4(v[r][4], v[r][5], v[r][6], v[r][7]);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; r++) {
    if (ta[r]) atomicAdd(&sthr[r], ta[r]);
    if (nz[r]) atomicAdd(&snum[r], nz[r]);
  }
  __syncthreads();
  if (tid < 4) {
    // (sum |w| 2^-35 + 2^16 sum over the small ones of 2^-24) / (nonzero weights 2^-25): 0 for a row
    // of zeros
    const float f = tid == 0 ? fac[0] : tid == 1 ? fac[1] : tid == 2 ? fac[2] : fac[3];
    const int rw = tid == 0 ? row[0] : tid == 1 ? row[1] : tid == 2 ? row[2] : row[3];
    const float thr = snum[tid] ? (float) sthr[tid] * (1.0f / 1024) / (float) snum[tid] : 0.0f;
    dst[2 * wn + Mp + rw] = f == f ? thr : __builtin_inff();
  }
}

// the largest of the 32 thresholds of a row block; thr: the rows' thresholds, the results behind them
__global__ void relayout_block_kernel(float *thr, int mt) {
  const int mb = blockIdx.x * blockDim.x + threadIdx.x;
  if (mb >= mt) return;
  float m = 0.0f;
  for (int r = 0; r < 32; r++) m = fmaxf(m, thr[mb * 32 + r]);
  thr[mt * 32 + mb] = m;
}

static int relayout_il_ok(int M, int il, const char *who) {
  if (il != 0 && (il < 1 || M != 4 * il || il % 8 != 0)) {
    set_err("%s: phase interleave needs M = 4 x rows per phase, a multiple of 8 (M %d, rows per phase %d)", who, M, il);
    return 0;
  }
  return 1;
}

extern "C" int ptk_relayout_il(float *dst, const float *wp, int M, int K, int cin, int il, void *s) {
  if (!relayout_il_ok(M, il, "ptk_relayout_il")) return -1;
  hipLaunchKernelGGL(relayout_kernel, dim3((unsigned) ((M + 31) / 32 * 8)), dim3(RELAY_THREADS), 0,
                     (hipStream_t) s, dst, wp, M, K, cin, ptk_conv_cinp(cin), il);
  HCHK(hipGetLastError());
  const int mt = (M + 31) / 32;
  hipLaunchKernelGGL(relayout_block_kernel, dim3((unsigned) ((mt + 63) / 64)), dim3(64), 0, (hipStream_t) s,
                     dst + 2ll * (mt * 32) * K * ptk_conv_cinp(cin) + mt * 32, mt);
  HCHK(hipGetLastError());
  return 0;
}
extern "C" int ptk_relayout(float *dst, const float *wp, int M, int K, int cin, void *s) {
  return ptk_relayout_il(dst, wp, M, K, cin, 0, s);
}

// ------------------------------------------------------------------------------ fp16 expansion
// binary16 -> binary32 by its bit fields.  Every binary16 value is exact in binary32: normals
// rebias the exponent (15 -> 127), subnormals m * 2^-24 renormalise around their leading one,
// inf / NaN keep sign and payload.  Integer work only, so no float mode (denormal flushing,
// NaN quieting) can change a result.
__device__ __forceinline__ unsigned half_to_float_bits(unsigned h) {
  const unsigned s = (h & 0x8000u) << 16, e = (h >> 10) & 0x1fu, m = h & 0x3ffu;
  if (e == 31u) return s | 0x7f800000u | (m << 13);
  if (e != 0u) return s | ((e + 112u) << 23) | (m << 13);
  if (m == 0u) return s;
  const unsigned p = 31u - (unsigned) __builtin_clz(m);   // leading one at bit p (0..9)
  return s | ((p + 103u) << 23) | ((m << (23u - p)) & 0x7fffffu);
}

__global__ void h2f_kernel(float *__restrict__ dst, const unsigned short *__restrict__ src,
                           long long n) {
  const long long st = (long long) gridDim.x * blockDim.x;
  for (long long i = (long long) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += st)
    dst[i] = __uint_as_float(half_to_float_bits(src[i]));
}

extern "C" int ptk_h2f(float *dst, const uint16_t *src, int64_t n, void *s) {
  if (n <= 0) return 0;
  long long blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(h2f_kernel, dim3((unsigned) blocks), dim3(256), 0, (hipStream_t) s, dst,
                     (const unsigned short *) src, (long long) n);
  HCHK(hipGetLastError());
  return 0;
}

// ------------------------------------------------------------------------------ epilogue
__device__ __forceinline__ float epi_apply(float v, const ptk_epi &e, int b, int co, long long col) {
  switch (e.op) {
    case PTK_EPI_LEAKY: return v >= 0.0f ? v : e.a * v;
    case PTK_EPI_RELU: return v > 0.0f ? v : 0.0f;
    case PTK_EPI_MULS: return v * e.a;
    case PTK_EPI_ADDS: return v + e.a;
    case PTK_EPI_ADDT: return v + e.t[(long long) b * e.bst + (long long) co * e.ldt + col];
    case PTK_EPI_DIVS: return v / e.a;
    default: return v;
  }
}

// input transform applied as a window element is staged (the reference's separate LeakyReLU node
// in front of a conv, fused): IN is a PTK_IN_* code.
// LeakyReLU as max(v, a*v): identical to (v >= 0 ? v : a*v) for 0 <= a <= 1 (signed zeros
// included), which the launcher enforces, in two instructions instead of three.
template <int IN>
__device__ __forceinline__ float in_xform(float v, float a) {
  if constexpr (IN != PTK_IN_PLAIN) v = fmaxf(v, a * v);
  return v;
}

// ------------------------------------------------------------------------------ MFMA conv kernel
// n / d for 0 <= n < 2^24 as (n * m) >> s, m = ceil(2^s / d), s = 24 + ceil(log2 d): the error
// term n * (m*d - 2^s) / (d * 2^s) stays below 1/d, so the floor is exact.  With n, m and s
// wave-uniform the division is two scalar multiplies and a shift.
struct FastDiv {
  unsigned m;
  int s;
};
static FastDiv fast_div(unsigned d) {
  int l = 0;
  while ((1u << l) < d) l++;
  const int s = 24 + l;
  return FastDiv{(unsigned) (((1ull << s) + d - 1) / d), s};
}
__device__ __forceinline__ int fdiv(int n, FastDiv f) {
  return (int) (((unsigned long long) (unsigned) n * f.m) >> f.s);
}

// Per-problem launch facts computed on the host: what a workgroup needs up to its first loads, in
// 32 bits and in one batch of scalar loads at kernel entry.
struct ConvProb {
  int count;                      // workgroups of the problem (grid row blockIdx.y = problem)
  int mt;                         // 32-row blocks
  int mtnt, mtnt0;                // mt x column tiles of a middle batch item / of item 0 (its columns
                                  // start ext_l earlier; one item: all of them)
  int last;                       // batch items - 1
  FastDiv div_tiles;              // by mtnt
  FastDiv div_mt;                 // by mt
  FastDiv div_phase;              // by C4 / 32 (row blocks per convT phase) when one_phase, else 0
  int flags;                      // PROB_*
  int ext_l;                      // item 0's first column is q0 - ext_l
  int addt;                       // the chain's first tensor add, or -1
  int M;                          // GEMM rows
  int q0;
  const void *x;                  // what the windows are loaded from (ptk_conv_desc x or xsp)
  const void *w;                  // fp16 weights
  const float *scale;             // their row factors
  const float *bias;
  int nbias4;                     // bytes of the bias
  int C4;
  int K, dil, st, cin, nchunk, ldx4, lim, shift;   // ldx4: input row stride in bytes
  long long bsx;
  int kd, xw;                     // (K - 1) * dil; window columns
  float in_a;
  int wslots;                     // ConvGroup's: LDS of one wave, in 16-byte slots
  int qend, ext_r;                // a middle item's column end; the last item's goes ext_r further
  int pad[6];
};
// every row block lies inside one phase (conv, or C4 % 32 == 0)
#define PROB_ONE_PHASE 1
// output / residual index ranges fit the 32-bit epilogue
#define PROB_FAST 2
// stride-4 convT with its rows interleaved by phase (row m: phase (m >> 3) & 3 of channel
// (m >> 5) * 8 + (m & 7))
#define PROB_PHASE_IL 4
// virtual input column 0 reads column 1, column c > 0 reads column c - 1
#define PROB_REFLECT 8
static_assert(sizeof(ConvProb) == 192, "three 64-byte scalar loads");

// What the fast epilogue reads, 128 bytes per problem, fetched in one batch of scalar loads when
// the epilogue starts (field by field from the descriptor, each chain op's fields had been a
// scalar load and a wait of their own).
struct ConvEpi {
  const float *y, *y2, *t;        // output, its LeakyReLU copy (or null), the residual of op addt
  const void *ysp;                // its LeakyReLU copy as split planes (or null)
  long long bsy, bst;             // batch strides of y / y2 and of t
  int ldy, ldt;                   // row strides (fit 32 bits on the fast path)
  int lout, qend, ext_r, ys, ypad, C4, nepi;   // qend: a middle item's column end
  int ops;                        // op e in bits 4e .. 4e + 3
  float a[PTK_MAX_EPI];
  float a2;
  int pad[5];
};
static_assert(sizeof(ConvEpi) == 128, "two 64-byte scalar loads");

struct ConvGroup {
  ConvProb info[PTK_MAX_GROUP];
  ConvEpi ep[PTK_MAX_GROUP];
  ptk_conv_desc d[PTK_MAX_GROUP];
  int ngroup;
  int wslots;                     // LDS of one wave, in 16-byte slots
  int wcols;                      // window columns staged (32 * units)
};

// Staged input window of one chunk (16 channels): NB column blocks of 32 outputs need
// (32*NB - 1)*stride + |K-1|*|dil| + 1 columns, staged as NU units of 32 columns (NU <= 4).  LDS
// holds it as planes [part][h] of 16-byte columns: plane (part, h), column c = that part of
// channels 8h .. 8h + 7.  The B operand a lane (column, h) needs for one tap and part is then one
// 16-byte LDS read, and each half-wave reads (and each staging store writes) consecutive 16-byte
// columns: no bank conflicts.
#define CONV_NU_MAX 4
// 16-byte LDS slots of one wave: its window / its partial sums
static constexpr int conv_slots(int nu, int nb) { return nu * 32 * 4 > nb * 256 ? nu * 32 * 4 : nb * 256; }
// and of the workgroup: flags, and one word per window column
#define CONV_EXTRA_SLOTS (2 + CONV_NU_MAX * 8)

// word 3 of a raw buffer resource on gfx9-family parts (gfx950): 32-bit data, range checked
#define PTK_BUF_WORD3 0x00020000
// an offset past every buffer: the load returns 0 (buffer range checking)
#define PTK_OOB 0x80000000u

// Scheduling fence for global loads: every instruction class except vector-memory may be moved
// across it (ALU, VALU, SALU, MFMA, LDS).  Placed right after prefetch loads, it keeps the machine
// scheduler from sinking them towards their use, which it does to shorten register live ranges
// and which would leave no prefetch distance at all.
#define PTK_PIN_VMEM() __builtin_amdgcn_sched_barrier(0x0106)

// voff: per-lane byte offset (PTK_OOB for an element that must read 0); soff: wave-uniform byte
// offset.  Either placement of the range check (with or without soff) leaves PTK_OOB + soff out of
// range for the buffers used here, which stay below 2 GiB.
__device__ __forceinline__ float buf_load(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

// the two parts of one lane's A or B operand
struct Parts {
  f16x8 h, l;
};

// min(m, |a|, |b|); NaN if any of them is
__device__ __forceinline__ float min_mag(float m, float a, float b) {
  asm("v_minimum3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(a), "v"(b));
  return m;
}

// Workgroups since the library was loaded that left outputs to the second pass / that ran it, the
// others having found nothing but exact zeros (counted on those rare paths only).
__device__ unsigned long long conv_stat[2];

// One workgroup = S waves on one block of 32 rows x 32*NB columns.  The waves take disjoint runs of
// the 16-channel chunks and are reduced through LDS in wave order (deterministic).  Each product of
// two fp32 values is taken as three fp16 products on v_mfma_f32_32x32x16_f16 (wl.xh, wh.xl, wh.xh:
// "weight relayout" above), accumulated in fp32.
//
// What an fp32 sum keeps is kept: with A = sum of |w x| over an output's products and n the nonzero
// weights of its row, the operands' parts cost at most (n/2 + 8) 2^-24 A on top of the sum's own
// rounding, whatever the magnitudes.  8 is the relative part.  The absolute parts, at most
// sum |w| 2^-35 + 2^-8 per small weight in scaled units, have to be below n 2^-25 A.  A is at least the
// sum over the waves of their partial sums' magnitudes: an output for which that is below its row's
// threshold, or NaN (an input past 2^(16 - CONV_XS) makes it that, as inf and NaN do), is left over.
// Ordinary outputs are not: all S partial sums would have to fall below about 2^-17 of their spread,
// which for inputs N(0, s) some 1e-11 / s^2 of them do (S = 2, C 128, K 3).  Each wave looks at its
// own partial sums first: in which eight rows of a column block is the smallest below the row block's
// largest threshold?  Only a workgroup whose waves all name the same judges its outputs one by one,
// one in a thousand of that launch.  (Judging every output and a barrier for the verdict took 0.3 us
// of each launch.)
//
// Where outputs are left, the block is computed by a second pass on v_mfma_f32_32x32x2_f32, from the
// fp32 operands, and they are stored from that: four rows of one lane together, so which pass an
// output comes from depends on its own receptive field and the four rows' weights, not on the tile
// or batch it is computed in.  Outputs that see nothing but zeros are left too, and skip that pass.
//
// Against a floor of 552 TFLOP/s of fp32 products (the fp16 rate the card sustains; 150 on the fp32
// matrix cores) it is bound by the way in and out of a workgroup (first loads, partial sums, stores),
// at batch 8 by operand loads as well: the matrix cores are 13-17 % busy in a T 226 decode's MRF
// launches, 37-45 % in eight of them (rocprofv3).  Against the fp32-MFMA kernel it replaced, us: MRF-256
// stack at T 904 149 -> 89, MRF-128 at T 3616 154 -> 109, conv_pre at T 226 6.3 -> 5.8, ups.0 11.4 ->
// 9.7, a T 226 decode 345 -> 241 and eight in a batch 2167 -> 1030; errors against 64 bits 0.36-0.90 of
// what they were on N(0, 1).  Inputs past 2^12, whose outputs take both passes: MRF-256 320-330, a T 226
// decode 810-880.
//
// KT: the taps the straight-line bodies are built for (11: K = 11, 7 and 3; 4: K = 4, the convT
// phase form); any other K goes through a rolled loop.  IN: input transform (PTK_IN_*).
template <int KT, int NB, int IN, int S>
__global__ void __launch_bounds__(64 * S) __attribute__((amdgpu_waves_per_eu(NB == 1 ? CONV_WPE1 : CONV_WPE2)))
conv_mfma_kernel(const ConvGroup g) {
  extern __shared__ u32x4 smem[];
  // Grid row blockIdx.y is the problem, so every field of it can be fetched at entry; rows are
  // as long as the largest problem's workgroup count, and the excess of a shorter one exits.
  const int p = blockIdx.y;
  const ConvProb pi = g.info[p];
  // (a field of each scalar-cache line, so that all loads go out together, ahead of the test)
  asm volatile("" ::"s"(pi.count), "s"(pi.x), "s"(pi.nbias4), "s"(pi.shift), "s"(pi.bsx), "s"(pi.kd), "s"(pi.wslots), "s"(pi.ext_r));
  const int bid = blockIdx.x, wslots = pi.wslots;
  if (bid >= pi.count) return;
  // Tiles item after item, column tile after column tile, row block fastest: item 0 has its own
  // number of column tiles, the last one takes the extra ones.  Written as masks and min / max
  // rather than selects, which the compiler turns into branches around the divisions (measured
  // slower on single-wave-per-SIMD launches).
  const int t = bid - pi.mtnt0;
  const int past0 = ~(t >> 31);                          // -1 past item 0's tiles, else 0
  const int bq = fdiv(max(t, 0), pi.div_tiles);
  const int b = min(bq + 1, pi.last) & past0;            // the last item takes its extra tiles
  const int r = bid - ((pi.mtnt0 + (b - 1) * pi.mtnt) & past0);
  const int tn = fdiv(r, pi.div_mt);
  const int mb = r - tn * pi.mt;
  const bool last_item = b == pi.last;
  const int q0 = pi.q0 - (pi.ext_l & ~past0) + tn * (32 * NB);   // this block's first column

  const int K = pi.K, dil = pi.dil, st = pi.st, cin = pi.cin, nchunk = pi.nchunk, lim = pi.lim;
  const unsigned ldx4 = (unsigned) pi.ldx4;
  const float in_a = pi.in_a;

  const int lane = threadIdx.x & 63;
  // wave index: uniform across the wave, which the compiler cannot see on its own (without this
  // the wave-based buffer resources would be treated as divergent)
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int chunk0 = w * nchunk / S, nch = (w + 1) * nchunk / S - chunk0;   // chunks of this wave
  // The phase of this row block (convT: row m is phase m / C4 of channel m % C4), when the block
  // lies inside one phase.
  const bool one_phase = (pi.flags & PROB_ONE_PHASE) != 0;
  // rows interleaved by phase: only the 4-tap convT phase form (KT = 4) carries that code (the
  // launcher refuses it elsewhere)
  const bool phase_il = KT == 4 && (pi.flags & PROB_PHASE_IL) != 0;
  const int r_tile = fdiv(mb, pi.div_phase);
  const int half = lane >> 5;     // which eight of a chunk's channels this lane feeds
  const int l32 = lane & 31;
  const int dmin = min(pi.kd, 0);
  const int XW = pi.xw;
  const int cmin = q0 * st + dmin - pi.shift;   // the window's first virtual column
  // Columns from here on are staged as zeros: past the row, past the window, or read by no output
  // of this item.  The last tile of an item rounds up past its columns, and in a launch over part
  // of the columns what lies there may never have been written.
  const int cend = max(min(lim, (min(q0 + 32 * NB, pi.qend + (last_item ? pi.ext_r : 0)) - 1) * st +
                                    max(pi.kd, 0) - pi.shift + 1), 0);
  u32x4 *const xs = smem + w * wslots;   // this wave's staging planes

  // Window columns this lane stages, fixed for the wave: unit u, column 32u + l32, channels 8*half
  // .. 8*half + 7 of the chunk; byte offset of the first, or an offset the buffer range check turns
  // into 0 (columns outside [0, cend)).  The row step and the chunk are wave-uniform
  // and go into the scalar offset.
  const long long xoff = b * pi.bsx;
  const unsigned nrec = (unsigned) cin * ldx4;
  unsigned voff[CONV_NU_MAX];
  {
    constexpr unsigned CB = IN == PTK_IN_SPLIT ? 16 : 4;   // bytes of a column of a row (or row group)
    const unsigned h8 = half ? 8u * ldx4 : 0u;
    int c = cmin + l32;
    if (pi.flags & PROB_REFLECT) {   // (column 0 reads column 1: the window holds 0 and 1 together)
#pragma unroll
      for (int u = 0; u < CONV_NU_MAX; u++, c += 32)
        voff[u] = (unsigned) c < (unsigned) cend ? (unsigned) (c == 0 ? 1 : c - 1) * CB + h8 : PTK_OOB;
    } else {
#pragma unroll
      for (int u = 0; u < CONV_NU_MAX; u++, c += 32)
        voff[u] = (unsigned) c < (unsigned) cend ? (unsigned) c * CB + h8 : PTK_OOB;
    }
  }

  float thr_b = 0.0f;   // the row block's largest threshold
  // accumulators: one 32x32 block per column block (16 values per lane)
  f32x16 acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; nb++)
#pragma unroll
    for (int v = 0; v < 16; v++) acc[nb][v] = 0.0f;

  // A operands: the wave's (chunk, tap) slices are contiguous, read through a buffer resource based
  // at its first chunk: the lane offset is fixed and the slice offset is wave-uniform, so a load
  // costs no vector address arithmetic
  const char *wbase = reinterpret_cast<const char *>(pi.w) +
                      (long long) (mb * nchunk + chunk0) * (K * CONV_TAPB);
  // (a resource with no records reads 0 and fetches nothing: the loads past the wave's last chunk)
  auto w_rsrc = [&](bool live) {
    return __builtin_amdgcn_make_buffer_rsrc(
        (void *) wbase, (short) 0, live ? (int) ((unsigned) K * (unsigned) nch * (unsigned) CONV_TAPB) : 0,
        PTK_BUF_WORD3);
  };
  auto x_rsrc = [&](bool live) {
    return __builtin_amdgcn_make_buffer_rsrc((void *) (reinterpret_cast<const float *>(pi.x) + xoff),
                                             (short) 0, live ? (int) nrec : 0, PTK_BUF_WORD3);
  };
  const unsigned wlane = (unsigned) lane * 16u;
  auto wa = [&](__amdgpu_buffer_rsrc_t rw, int slice) {
    const int so = slice * CONV_TAPB;
    Parts a;
    a.h = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(rw, wlane, so, 0));
    a.l = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(rw, wlane + 1024u, so, 0));
    return a;
  };

  // The chunk loop, for a compile-time tap count KC (0: runtime K) and NU window units.  A chunk's
  // window goes through three stages: its loads are issued while the chunk two before it runs, its
  // split (32 VALU instructions a unit) runs between the MFMAs of the chunk before it, which hide up
  // to six VALU instructions each (measured: 12 MFMAs 181 ns, with 72 VALU between them 185 ns), and
  // only the LDS stores stand between two chunks.  Rows past cin exist only when cin is not a
  // multiple of 16; MASK (compile time) selects the code that handles them.
  auto run = [&](auto kc, auto mask, auto nuc) {
    constexpr int KC = decltype(kc)::value, NU = decltype(nuc)::value;
    constexpr bool MASK = decltype(mask)::value;
    constexpr int PS = NU * 32;   // plane stride (16-byte slots)
    constexpr int PDM = NB == 1 ? CONV_PD1 : CONV_PD2, PD = KC == 0 ? 1 : KC < PDM ? KC : PDM;   // slices A is loaded ahead
    constexpr bool SPLIT = IN == PTK_IN_SPLIT;
    float raw[NU][8];               // fp32 input: what is loaded
    u32x4 raws[NU][2];              // split planes: what is loaded
    u32x4 sp[NU][2];
    auto load_unit = [&](__amdgpu_buffer_rsrc_t rx, int u, int j) {
      const int ci0 = (chunk0 + j) * CONV_CK;
      if constexpr (SPLIT) {
        const unsigned so = (unsigned) ci0 * ldx4;
        raws[u][0] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, voff[u], so, 0));
        raws[u][1] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, voff[u], so + 4u * ldx4, 0));
        return;
      }
#pragma unroll
      for (int r = 0; r < 8; r++) {
        if constexpr (MASK) {   // a row past cin reads 0
          const unsigned vo = voff[u] != PTK_OOB && ci0 + 8 * half + r < cin
              ? voff[u] + (unsigned) (ci0 + r) * ldx4 : PTK_OOB;
          raw[u][r] = buf_load(rx, vo, 0);
        } else {
          raw[u][r] = buf_load(rx, voff[u], (unsigned) (ci0 + r) * ldx4);
        }
      }
    };
    auto split_unit = [&](int u, int e) {   // channels 2e, 2e + 1 of this lane's eight
      if constexpr (SPLIT) {
        sp[u][0][e] = raws[u][0][e];
        sp[u][1][e] = raws[u][1][e];
        return;
      }
      const float a = in_xform<IN>(raw[u][2 * e], in_a), b = in_xform<IN>(raw[u][2 * e + 1], in_a);
      unsigned h, l;
      split_input(a, b, h, l);
      sp[u][0][e] = h;
      sp[u][1][e] = l;
    };
    auto store_window = [&]() {
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int u = 0; u < NU; u++)
#pragma unroll
        for (int q = 0; q < 2; q++) xs[half * PS + 2 * q * PS + 32 * u + l32] = sp[u][q];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    const int sc = KC > 0 ? 1 : st;   // the straight-line bodies take stride 1 only
    const u32x4 *const xl = xs + half * PS + l32 * sc - dmin;   // tap 0, column block 0
    auto col = [&](int k, int nb) {   // B operands of tap k, column block nb
      const u32x4 *xr = xl + k * dil + 32 * nb * sc;
      Parts q;
      q.h = __builtin_bit_cast(f16x8, xr[0]);
      q.l = __builtin_bit_cast(f16x8, xr[2 * PS]);
      return q;
    };
    auto mfma3 = [&](const Parts &a, const f16x8 &hs, const Parts &c, int nb) {
      acc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hs, c.l, acc[nb], 0, 0, 0);
      acc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.l, c.h, acc[nb], 0, 0, 0);
      acc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.h, c.h, acc[nb], 0, 0, 0);
    };
    const __amdgpu_buffer_rsrc_t rx = x_rsrc(true), rw = w_rsrc(true);
    const int last = nch * K - 1;   // the wave's last slice
    Parts ahead[PD];
#pragma unroll
    for (int u = 0; u < NU; u++) load_unit(rx, u, 0);
#pragma unroll
    for (int k = 0; k < PD; k++) ahead[k] = wa(rw, min(k, last));
    // (a vector load, in line behind those that the loop waits for; a scalar one would hold up its
    // first LDS reads)
    thr_b = buf_load(__builtin_amdgcn_make_buffer_rsrc((void *) (pi.scale + pi.mt * 64), (short) 0, pi.mt * 4, PTK_BUF_WORD3), 0,
                     (unsigned) mb * 4u);
    {
      const __amdgpu_buffer_rsrc_t rx1 = x_rsrc(nch > 1);
#pragma unroll
      for (int u = 0; u < NU; u++) {
#pragma unroll
        for (int e = 0; e < 4; e++) split_unit(u, e);
        load_unit(rx1, u, 1);
      }
    }
    for (int j = 0; j < nch; j++) {
      store_window();
      const __amdgpu_buffer_rsrc_t rx2 = x_rsrc(j + 2 < nch);
      if constexpr (KC > 0) {
        // Steps of three MFMAs, (tap, column block).  A step's B operands are read while the step
        // before it runs; the scheduling barrier keeps the compiler from reading further ahead,
        // which would take more registers than there are.
        constexpr int NS = KC * NB, S0 = NS / 3, NP = NU * 4;
        Parts a[KC + PD];
#pragma unroll
        for (int k = 0; k < PD; k++) a[k] = ahead[k];
        constexpr int LA = NB == 1 ? CONV_LA1 : CONV_LA2;   // steps the B operands are read ahead
        Parts q[NS + LA];
        f16x8 hs;   // a[k].h shifted to the lo's scale
#pragma unroll
        for (int s = 0; s < LA; s++) q[s] = col(s / NB, s % NB);
#pragma unroll
        for (int s = 0; s < NS; s++) {
          const int k = s / NB, nb = s % NB;
          if (s + LA < NS) q[s + LA] = col((s + LA) / NB, (s + LA) % NB);
          if (nb == 0) a[k + PD] = wa(rw, k + PD < KC ? j * KC + k + PD : min(j * KC + k + PD, last));
          // the next chunk's split over the last two thirds of the steps
#pragma unroll
          for (int i = 0; i < NP; i++)
            if (S0 + i * (NS - S0) / NP == s) {
              split_unit(i / 4, i % 4);
              if (i % 4 == 3) load_unit(rx2, i / 4, j + 2);
            }
          if (nb == 0) hs = a[k].h * (_Float16) (1.0f / CONV_LS);
          mfma3(a[k], hs, q[s], nb);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int k = 0; k < PD; k++) ahead[k] = a[KC + k];
      } else {
        for (int k = 0; k < K; k++) {
          const Parts a = ahead[0];
          ahead[0] = wa(rw, min(j * K + k + 1, last));
          PTK_PIN_VMEM();
#pragma unroll
          for (int nb = 0; nb < NB; nb++) mfma3(a, a.h * (_Float16) (1.0f / CONV_LS), col(k, nb), nb);
        }
#pragma unroll
        for (int u = 0; u < NU; u++) {
#pragma unroll
          for (int e = 0; e < 4; e++) split_unit(u, e);
          load_unit(rx2, u, j + 2);
        }
      }
    }
  };
  // The second pass: the same chunks from fp32 operands, in one rolled loop; the loads of a chunk's
  // window go out ahead of the taps of the chunk before it, those of a tap's weights ahead of the tap
  // before it.  The window is staged as planes [h][e >> 2] of float4 columns (channels 8h + e): the
  // same LDS.  pi, p: the launch facts, read again (kept from the first pass they would take the
  // scalar registers of the common path).
  // the input transform as the fp32 operands need it: split planes hold LeakyReLU(in_a) of d.x
  auto xform32 = [&](float v, float a) {
    return in_xform<IN == PTK_IN_PLAIN ? PTK_IN_PLAIN : PTK_IN_LEAKY>(v, a);
  };
  auto run32 = [&](const ConvProb &pi, int p) {
    const ptk_conv_desc &d = g.d[p];
    const int PS = g.wcols, K = pi.K, dil = pi.dil, st = pi.st, cin = pi.cin, nchunk = pi.nchunk;
    const unsigned ldx4 = (unsigned) pi.ldx4;
    const float in_a = pi.in_a;
    const int chunk0 = w * nchunk / S, nch = (w + 1) * nchunk / S - chunk0;
    if (nch == 0) return;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        (void *) (d.x + b * pi.bsx), (short) 0, (int) ((unsigned) cin * ldx4), PTK_BUF_WORD3);
    const float4 *const wr = reinterpret_cast<const float4 *>(d.w + (long long) (pi.mt * 32) * K * d.cinp) +
                             ((long long) mb * nchunk + chunk0) * K * (CONV_TAPB / 16) + lane * 2;
    float4 *const x4 = reinterpret_cast<float4 *>(xs);
    float raw[CONV_NU_MAX][8];
    auto load = [&](int j) {
      const int ci0 = (chunk0 + j) * CONV_CK + 8 * half;
#pragma unroll
      for (int u = 0; u < CONV_NU_MAX; u++) {
        if (32 * u >= PS) continue;
        const unsigned c4 = IN == PTK_IN_SPLIT ? (voff[u] - (unsigned) (8 * half) * ldx4) / 4u
                                               : voff[u] - (unsigned) (8 * half) * ldx4;
#pragma unroll
        for (int e = 0; e < 8; e++)
          raw[u][e] = buf_load(rx, j < nch && voff[u] != PTK_OOB && ci0 + e < cin
                                       ? c4 + (unsigned) (ci0 + e) * ldx4 : PTK_OOB, 0);
      }
    };
    load(0);
    float4 a0 = wr[0], a1 = wr[1];
    for (int j = 0; j < nch; j++) {
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int u = 0; u < CONV_NU_MAX; u++) {
        if (32 * u >= PS) continue;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = xform32(raw[u][e], in_a);
        x4[2 * half * PS + 32 * u + l32] = make_float4(v[0], v[1], v[2], v[3]);
        x4[(2 * half + 1) * PS + 32 * u + l32] = make_float4(v[4], v[5], v[6], v[7]);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      load(j + 1);
      PTK_PIN_VMEM();
      for (int k = 0; k < K; k++) {
        const float4 *const wk = wr + (long long) min(j * K + k + 1, nch * K - 1) * (CONV_TAPB / 16);
        const float4 n0 = wk[0], n1 = wk[1];
        PTK_PIN_VMEM();
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
          const float4 *const xr = x4 + 2 * half * PS + (l32 + 32 * nb) * st - min((K - 1) * dil, 0) + k * dil;
          const float4 b0 = xr[0], b1 = xr[PS];
          acc[nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.x, b0.x, acc[nb], 0, 0, 0);
          acc[nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.y, b0.y, acc[nb], 0, 0, 0);
          acc[nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.z, b0.z, acc[nb], 0, 0, 0);
          acc[nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.w, b0.w, acc[nb], 0, 0, 0);
          acc[nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.x, b1.x, acc[nb], 0, 0, 0);
          acc[nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.y, b1.y, acc[nb], 0, 0, 0);
          acc[nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.z, b1.z, acc[nb], 0, 0, 0);
          acc[nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.w, b1.w, acc[nb], 0, 0, 0);
        }
        a0 = n0;
        a1 = n1;
      }
    }
  };
  constexpr std::false_type nomask{};
  constexpr std::integral_constant<int, NB + 1> few{};
  constexpr std::integral_constant<int, CONV_NU_MAX> all{};
  const bool narrow = XW <= 32 * (NB + 1);
  // channel padding in the last chunk, a stride or another K: the rolled body
  const int straight = cin == nchunk * CONV_CK && st == 1 ? K : 0;
  if (nch == 0) {}
  else if (KT == 4 && straight == 4 && narrow) run(std::integral_constant<int, KT == 4 ? 4 : 0>{}, nomask, few);
  else if (KT == 11 && straight == 11 && narrow) run(std::integral_constant<int, KT == 11 ? 11 : 0>{}, nomask, few);
  else if (KT == 11 && straight == 11) run(std::integral_constant<int, KT == 11 ? 11 : 0>{}, nomask, all);
  else if (KT == 11 && straight == 7 && narrow) run(std::integral_constant<int, KT == 11 ? 7 : 0>{}, nomask, few);
  else if (KT == 11 && straight == 3 && narrow) run(std::integral_constant<int, KT == 11 ? 3 : 0>{}, nomask, few);
  else run(std::integral_constant<int, 0>{}, std::true_type{}, all);

  // Epilogue: the S partial sums of a block are added in wave order through LDS, then bias, the
  // epilogue chain and one store per output.  Lane (l32, half) holds, for column block nb, the 16
  // values v of column q0 + 32*nb + l32 at rows 8*(v >> 2) + 4*half + (v & 3) of the block.  Wave w
  // finishes the NMAX = 16 / S values from v0 = w * NMAX, in groups of GRP = 4 (rows of one v >> 2).
  constexpr int NMAX = 16 / S, GRP = 4, NG = NMAX / GRP;
  const int v0 = w * NMAX;
  const int addt = pi.addt;   // the chain's residual add, if any
  auto vrow = [&](int i) { return 8 * ((v0 + i) >> 2) + 4 * half + ((v0 + i) & 3); };   // of value i
  // bit nb * NG + gg: outputs of group gg, column block nb, that the first pass leaves
  unsigned left = 0;
  int *const flags = reinterpret_cast<int *>(smem + S * wslots);
  bool nonzero = false;   // some partial sum of theirs is not zero, or their row has no fp16 form
  bool judged = false;    // the workgroup judged its outputs
  // (once for each pass, not a loop over them: the compiler would compute everything the rare paths
  // need ahead of the loop, some 200 instructions)
  auto finish = [&](auto passc, const ConvProb &pi, int p) {
  constexpr int pass = decltype(passc)::value;
  const ptk_conv_desc &d = g.d[p];
  // Each wave writes its partial sums over its own staging area, which only it reads, so no wave
  // waits for the others before writing: [nb][v >> 2][lane] float4.
  {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    f32x4 *red = reinterpret_cast<f32x4 *>(xs);
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        f32x4 v;
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = acc[nb][4 * q + i];
        red[(nb * 4 + q) * 64 + lane] = v;
      }
  }
  // A wave's look at its own partial sums (while the epilogue's loads are on their way) and the barrier
  // behind them.  Returns what the waves say, read together with the first sums.
  auto reduce_wait = [&]() {
    if (pass != 0) {
      __syncthreads();
      return 0;
    }
    const int qend = pi.qend + (last_item ? pi.ext_r : 0);
    unsigned low = 0;   // bit 4 * nb + (v >> 2): rows 8 * (v >> 2) .. + 7 of column block nb
    unsigned long long used[NB], any = 0;
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      float m = __builtin_inff();
#pragma unroll
      for (int v = 0; v < 16; v += 2) m = min_mag(m, acc[nb][v], acc[nb][v + 1]);
      used[nb] = __ballot(q0 + 32 * nb + l32 < qend);
      any |= __ballot(!(m >= thr_b)) & used[nb];
    }
    if (any != 0) {   // (a few in a hundred of a large launch's waves)
      float all = 0.0f;
#pragma unroll
      for (int nb = 0; nb < NB; nb++)
#pragma unroll
        for (int v = 0; v < 16; v += 4) {
          const float m = min_mag(min_mag(__builtin_inff(), acc[nb][v], acc[nb][v + 1]), acc[nb][v + 2], acc[nb][v + 3]);
          all = min_mag(all, m, m);
          low |= (__ballot(!(m >= thr_b)) & used[nb]) != 0 ? 1u << (4 * nb + v / 4) : 0u;
        }
      const int rows = pi.M - mb * 32;   // (the padding rows behind them are all zero)
      low &= rows >= 32 ? 0xffu : 0x11u * ((1u << ((rows + 7) >> 3)) - 1);
      // a NaN makes the workgroup judge whatever the other waves have
      if (__ballot(all != all) != 0) low |= 0x100;
    }
    if (lane == 0) flags[w] = nch > 0 ? (int) low : 0xff;   // (a wave without channels has no say)
    if (threadIdx.x == 0) flags[4] = flags[5] = 0;
    __syncthreads();
    int all = flags[0], nan = all;
#pragma unroll
    for (int i = 1; i < S; i++) {
      all &= flags[i];
      nan |= flags[i];
    }
    return all | (nan & 0x100);
  };
  // The judging, if all waves ask for it.
  auto judge = [&](int say) {
    if (pass != 0 || __builtin_expect(__builtin_amdgcn_readfirstlane(say) == 0, 1)) return;
    judged = true;
    const int qend = pi.qend + (last_item ? pi.ext_r : 0);
    f32x4 thr[NG];
#pragma unroll
    for (int gg = 0; gg < NG; gg++)
      thr[gg] = *reinterpret_cast<const f32x4 *>(pi.scale + (pi.mt + mb) * 32 + vrow(gg * GRP));
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
#pragma unroll
      for (int gg = 0; gg < NG; gg++) {
        f32x4 m = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < S; i++)
          m += __builtin_elementwise_abs(reinterpret_cast<const f32x4 *>(smem + i * wslots)[(nb * 4 + (v0 >> 2) + gg) * 64 + lane]);
        bool ok = true, some = false;
#pragma unroll
        for (int e = 0; e < GRP; e++) {
          const bool is = m[e] >= thr[gg][e] && m[e] < __builtin_inff();
          ok &= is;
          some |= !is && (m[e] != 0.0f || thr[gg][e] == __builtin_inff());
        }
        const bool used = q0 + 32 * nb + l32 < qend;
        left |= (unsigned) (used && !ok) << (nb * NG + gg);
        nonzero |= used && some;
      }
  };
  // The S partial sums of a group's values, in wave order.
  auto reduced = [&](int nb, int gg) {
    const int v = v0 + gg * GRP;
    f32x4 part[S];
#pragma unroll
    for (int i = 0; i < S; i++)
      part[i] = reinterpret_cast<const f32x4 *>(smem + i * wslots)[(nb * 4 + (v >> 2)) * 64 + lane];
    f32x4 sum = part[0];
#pragma unroll
    for (int i = 1; i < S; i++) sum += part[i];
    return sum;
  };
  // Fast path: a full block whose rows are consecutive output channels (conv, or a convT block
  // inside one phase), with every index of the output, its LeakyReLU copy and the residual inside
  // 32 bits (the launcher checks the extents).  Addresses are a wave-uniform row offset, in the
  // scalar offset of a buffer access, plus a lane offset computed once per column; the residual
  // loads are issued before the reduction barrier, at a clamped column so that every lane loads
  // in bounds without a branch (a lane whose column does not exist stores nothing).  The chain runs
  // op by op over a lane's values, one branch per op.  A convT block with its rows interleaved by
  // phase (phase_il) holds 8 whole channels.
  // A partial block (the rows of a conv behind its last output) stores the groups that exist; its
  // bias reads 0 past the end, its scale is there for every row, a residual would not be.
  const bool part_block = mb * 32 + 32 > pi.M;
  if ((pi.flags & PROB_FAST) && (one_phase || phase_il) && (!part_block || (addt < 0 && pi.M == pi.C4 && pi.M % 4 == 0))) {
    const ConvEpi ep = g.ep[p];
    // first channel of the block
    const long long row0 = phase_il ? (long long) mb * 8 : (long long) mb * 32 - (long long) r_tile * ep.C4;
    const int ldy32 = ep.ldy, ldt32 = ep.ldt;
    float *yk = const_cast<float *>(ep.y) + (long long) b * ep.bsy + row0 * ldy32;
    const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(
        (void *) yk, (short) 0, (int) 0x7fffffff, PTK_BUF_WORD3);
    const __amdgpu_buffer_rsrc_t ry2 = __builtin_amdgcn_make_buffer_rsrc(
        (void *) (ep.y2 != nullptr ? ep.y2 + (long long) b * ep.bsy + row0 * ldy32 : yk), (short) 0,
        (int) 0x7fffffff, PTK_BUF_WORD3);
    const __amdgpu_buffer_rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(
        (void *) (addt >= 0 ? ep.t + (long long) b * ep.bst + row0 * ldt32 : yk), (short) 0,
        (int) 0x7fffffff, PTK_BUF_WORD3);
    const __amdgpu_buffer_rsrc_t rys = __builtin_amdgcn_make_buffer_rsrc(
        (void *) (ep.ysp != nullptr ? reinterpret_cast<const float *>(ep.ysp) + (long long) b * ep.bsy + row0 * ldy32 : yk),
        (short) 0, (int) 0x7fffffff, PTK_BUF_WORD3);
    // wave-uniform part of the row of value i (the lane part is 4 * half)
    auto urow = [&](int i) { return 8 * ((v0 + i) >> 2) + ((v0 + i) & 3); };
    const int qend32 = ep.qend + (last_item ? ep.ext_r : 0);
    const int rows = pi.M - mb * 32 - 4 * half;
    float rv[NB][NMAX];
    if (addt >= 0) {
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        const int q = q0 + 32 * nb + l32;
        const int col = q * ep.ys + r_tile - ep.ypad;
        const int cl = q < qend32 && col >= 0 && col < ep.lout ? col : 0;
#pragma unroll
        for (int i = 0; i < NMAX; i++)
          rv[nb][i] = buf_load(rt, (unsigned) (4 * half * ldt32 + cl) * 4u, (unsigned) (urow(i) * ldt32) * 4u);
      }
    }
    // the bias and scale of a lane's rows (a row without a bias is past the buffer and reads 0), in
    // flight with the residual while the partial sums are written
    f32x4 bias[NG], scale[NG];
    {
      const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *) pi.bias, (short) 0, pi.nbias4, PTK_BUF_WORD3);
#pragma unroll
      for (int gg = 0; gg < NG; gg++) {
        const int rg = urow(gg * GRP);
        bias[gg] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
            rb, (unsigned) ((int) row0 + 4 * half + (phase_il ? 0 : rg)) * 4u, 0, 0));
        if constexpr (pass == 0) scale[gg] = *reinterpret_cast<const f32x4 *>(pi.scale + mb * 32 + 4 * half + rg);
        else scale[gg] = f32x4{1.0f, 1.0f, 1.0f, 1.0f};
      }
    }
    const int say = reduce_wait();
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
      const int q = q0 + 32 * nb + l32;
      const int col = q * ep.ys + r_tile - ep.ypad;   // phase_il: the sample of phase 0 (r_tile = 0)
      const bool oq = q < qend32;
      float val[NMAX];
#pragma unroll
      for (int gg = 0; gg < NG; gg++) {
        const f32x4 sum = reduced(nb, gg);
#pragma unroll
        for (int i = 0; i < GRP; i++) val[gg * GRP + i] = fmaf(sum[i], scale[gg][i], bias[gg][i]);
      }
      if (nb == 0) judge(say);
      // The chain.  The decoder's two chains, a LeakyReLU and a tensor add (the chain's one, the
      // launcher's rule), have their own code; any other goes op by op.
      if (ep.ops == PTK_EPI_ADDT) {
#pragma unroll
        for (int i = 0; i < NMAX; i++) val[i] = val[i] + rv[nb][i];
      } else if (ep.ops == PTK_EPI_LEAKY) {
#pragma unroll
        for (int i = 0; i < NMAX; i++) val[i] = val[i] >= 0.0f ? val[i] : ep.a[0] * val[i];
      } else {
#pragma unroll 1
        for (int e = 0; e < ep.nepi; e++) {
          const int op = (ep.ops >> (4 * e)) & 15;
          const float a = e == 0 ? ep.a[0] : e == 1 ? ep.a[1] : e == 2 ? ep.a[2] : ep.a[3];
#pragma unroll
          for (int i = 0; i < NMAX; i++) {
            const float v = val[i];
            val[i] = op == PTK_EPI_LEAKY ? (v >= 0.0f ? v : a * v) : op == PTK_EPI_RELU ? (v > 0.0f ? v : 0.0f)
                   : op == PTK_EPI_MULS ? v * a : op == PTK_EPI_ADDS ? v + a : op == PTK_EPI_DIVS ? v / a
                   : op == PTK_EPI_ADDT ? v + rv[nb][i] : v;
          }
        }
      }
      // Stores by groups: four rows of one v >> 2.  Rows interleaved by phase: v >> 2 is
      // the phase, the column's sample.
#pragma unroll
      for (int gg = 0; gg < NG; gg++) {
        const int vg = v0 + gg * GRP;
        const int cg = phase_il ? col + (vg >> 2) : col;
        const int rg = phase_il ? (vg & 3) : urow(gg * GRP);   // uniform part of the group's first row
        if (!(oq && cg >= 0 && cg < ep.lout && 8 * (vg >> 2) < rows && (left >> (nb * NG + gg) & 1) == pass)) continue;
        const unsigned vo = (unsigned) (4 * half * ldy32 + cg) * 4u;
#pragma unroll
        for (int i = 0; i < GRP; i++) {
          const float v = val[gg * GRP + i];
          const unsigned so = (unsigned) ((rg + i) * ldy32) * 4u;
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), ry, vo, so, 0);
          if (ep.y2 != nullptr)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v >= 0.0f ? v : ep.a2 * v), ry2, vo, so, 0);
        }
        if (ep.ysp != nullptr) {
          // channel 4 * half + (rg & 3) of the eight-channel group rg >> 3, hi row then lo row
          unsigned h[GRP / 2], l[GRP / 2];
#pragma unroll
          for (int i = 0; i < GRP; i += 2) {
            const float a = val[gg * GRP + i], c = val[gg * GRP + i + 1];
            split_input(a >= 0.0f ? a : ep.a2 * a, c >= 0.0f ? c : ep.a2 * c, h[i / 2], l[i / 2]);
          }
          const unsigned vs = (unsigned) cg * 16u + (unsigned) half * 8u;
          const unsigned ss = (unsigned) ((rg >> 3) * 8 * ldy32) * 4u + (unsigned) (rg & 3) * 2u;
          typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
          __builtin_amdgcn_raw_buffer_store_b64(u32x2{h[0], h[1]}, rys, vs, ss, 0);
          __builtin_amdgcn_raw_buffer_store_b64(u32x2{l[0], l[1]}, rys, vs, ss + 16u * (unsigned) ldy32, 0);
        }
      }
    }
  } else {
  // General path (partial row blocks of a convT or with a residual, convT phases that straddle a
  // block, large tensors): per
  // element
  const int M = d.M, C4 = d.C4, ys = d.ys, ypad = d.ypad, nepi = d.nepi;
  const long long Lout = d.Lout, ldy = d.ldy;
  float *yb = d.y + (long long) b * d.bsy;
  float *y2b = d.y2 != nullptr ? d.y2 + (long long) b * d.bsy : nullptr;
  float *ysb = d.ysp != nullptr ? reinterpret_cast<float *>(d.ysp) + (long long) b * d.bsy : nullptr;
  const float a2 = d.a2;
  const bool phase_rows = C4 != M;
  const long long qend = d.q0 + d.nq + (last_item ? d.ext_r : 0);
  judge(reduce_wait());
#pragma unroll 1
  for (int nb = 0; nb < NB; nb++) {
    const long long q = (long long) q0 + 32 * nb + l32;
#pragma unroll 1
    for (int gg = 0; gg < NG; gg++) {
    const f32x4 sum = reduced(nb, gg);
#pragma unroll
    for (int i = 0; i < GRP; i++) {
      const int m = mb * 32 + vrow(gg * GRP + i);
      if (m >= M || q >= qend || (left >> (nb * NG + gg) & 1) != pass) continue;
      int co = m, r = 0;
      if (phase_il) {
        r = (m >> 3) & 3;
        co = (m >> 5) * 8 + (m & 7);
      } else if (phase_rows) {
        r = m / C4;
        co = m - r * C4;
      }
      const long long col = q * ys + r - ypad;
      if (col < 0 || col >= Lout) continue;
      float v = fmaf(sum[i], pass == 0 ? pi.scale[m] : 1.0f, d.bias != nullptr && co < d.nbias ? d.bias[co] : 0.0f);
      for (int e = 0; e < nepi; e++) v = epi_apply(v, d.epi[e], b, co, col);
      const long long yi = (long long) co * ldy + col;
      yb[yi] = v;
      const float vl = v >= 0.0f ? v : a2 * v;
      if (y2b != nullptr) y2b[yi] = vl;
      if (ysb != nullptr) {
        unsigned h, l;
        split_input(vl, 0.0f, h, l);
        unsigned short *const ys16 = reinterpret_cast<unsigned short *>(ysb + (long long) (co & ~7) * ldy) + col * 8 + (co & 7);
        ys16[0] = (unsigned short) h;
        ys16[8 * ldy] = (unsigned short) l;
      }
    }
    }
  }
  }
  };
  finish(std::integral_constant<int, 0>{}, pi, p);
  if (__builtin_expect(!judged, 1)) return;
  if (left) flags[4] = 1;
  if (nonzero) flags[5] = 1;
  __syncthreads();   // (every wave is done with the first pass's partial sums, too)
  if (__builtin_amdgcn_readfirstlane(flags[4]) == 0) return;
  if (threadIdx.x == 0) atomicAdd(&conv_stat[0], 1ull);
  int p2 = blockIdx.y;
  asm volatile("" : "+s"(p2));   // (so that the facts are read again, see run32)
  const ConvProb pr = g.info[p2];
  int again = __builtin_amdgcn_readfirstlane(flags[5]);
  if (again == 0) {
    // Sums of exactly zero: of nothing but zeros, or of values below the parts' range?  Threads take a
    // column each and share its channels.
    const ptk_conv_desc &d = g.d[p2];
    const int XW = pr.xw, K = pr.K, dil = pr.dil, st = pr.st, cin = pr.cin;
    const int dmin = min(pr.kd, 0), cmin = q0 * st + dmin - pr.shift;
    const int cend = min(pr.lim, (min(q0 + 32 * NB, pr.qend + (last_item ? pr.ext_r : 0)) - 1) * st + max(pr.kd, 0) - pr.shift + 1);
    int *const cm = flags + 8;   // per window column: it holds something
    const int cols = XW <= 64 ? 64 : 128, i = threadIdx.x & (cols - 1);
    for (int k = threadIdx.x; k < 32 * CONV_NU_MAX; k += 64 * S) cm[k] = 0;
    __syncthreads();
    const int c = cmin + i, pc = pr.flags & PROB_REFLECT ? (c == 0 ? 1 : c - 1) : c;
    if (i < XW && c >= 0 && c < cend) {
      bool any = false;
#pragma unroll 8
      for (int ci = threadIdx.x / cols; ci < cin; ci += 64 * S / cols)
        any |= xform32(d.x[b * pr.bsx + (long long) ci * d.ldx + pc], pr.in_a) != 0.0f;
      if (any) cm[i] = 1;
    }
    __syncthreads();
    int seen = 0;
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
      if (left >> (nb * NG) & ((1u << NG) - 1))
        for (int k = 0; k < K; k++) seen |= cm[(l32 + 32 * nb) * st - dmin + k * dil];
    if (seen) flags[5] = 1;
    __syncthreads();
    again = __builtin_amdgcn_readfirstlane(flags[5]);
  }
  // the outputs left over, from fp32 operands (zeros add up to what the first pass has: zero)
#pragma unroll
  for (int nb = 0; nb < NB; nb++)
#pragma unroll
    for (int v = 0; v < 16; v++) acc[nb][v] = 0.0f;
  if (again) {
    if (threadIdx.x == 0) atomicAdd(&conv_stat[1], 1ull);
    run32(pr, p2);
  }
  finish(std::integral_constant<int, 1>{}, pr, p2);
}

static int conv_window(const ptk_conv_desc *d, int nb) {
  const int kd = (d->K - 1) * d->dil;
  return (32 * nb - 1) * d->stride + (kd < 0 ? -kd : kd) + 1;
}

// Kernel-selection knobs (PTK_*), read from the environment once per process, at the first
// launch that consults them, not per launch: launches come from many serving threads at once, and
// getenv is neither cheap nor safe against a concurrent setenv.  ptk_knobs_reload re-reads them
// (tests that change a knob between calls); each is an atomic int, so a launch running meanwhile
// sees the old or the new value of each knob.
enum KnobId {
  KN_CONV_SPLIT, KN_CONV_NB, KN_CONV_FAST, KN_TAIL_OUT,
  KN_TAIL_GRID, KN_TAIL_XCD, KN_NARROW, KN_COUNT
};
static const struct {
  const char *name;
  int dflt;
} kKnobs[KN_COUNT] = {{"PTK_CONV_SPLIT", 0}, {"PTK_CONV_NB", 0}, {"PTK_CONV_FAST", 1},
                      {"PTK_TAIL_OUT", 0},
                      {"PTK_TAIL_GRID", 0},   {"PTK_TAIL_XCD", 1},  {"PTK_NARROW", 1}};
static std::atomic<int> g_knob[KN_COUNT];
static std::once_flag g_knob_once;
static std::mutex g_knob_lock;

static void knobs_read() {
  std::lock_guard<std::mutex> lk(g_knob_lock);
  for (int i = 0; i < KN_COUNT; i++) {
    const char *e = getenv(kKnobs[i].name);
    g_knob[i].store(e ? atoi(e) : kKnobs[i].dflt, std::memory_order_relaxed);
  }
}
static int knob(KnobId k) {
  std::call_once(g_knob_once, knobs_read);
  return g_knob[k].load(std::memory_order_relaxed);
}
extern "C" void ptk_knobs_reload(void) {
  std::call_once(g_knob_once, knobs_read);
  knobs_read();
}

// Tile shape: the channel split S in {2, 4} (PTK_CONV_SPLIT overrides) and the column blocks per
// wave NB in {1, 2} (PTK_CONV_NB).
// S fixes the order in which a block's partial sums are added, so it is chosen from one batch item's
// grid (of nq_shape columns when the launch covers a sub-range): a batched item's result is
// bit-identical to the same item alone.  Measured: S = 2 against 4 at C 128, T 3616, batch 8 159-165
// against 175-195 us, at C 256, T 904 37 against 30 us.
// NB changes no bit and is chosen from the whole launch.  Up to a few workgroups per CU a launch takes
// as long as its fullest CU, and a workgroup of two column blocks 1.2 to 1.4 times one of one block:
// two are worth it where they take a round of 256 workgroups less, and from 512 on, where every CU has
// several either way.  One against two blocks, us, S = 4: K 3, C 256, 232 / 120 workgroups 6.6 / 8.2,
// 408 / 208 9.0 / 8.3, 504 / 264 9.2 / 10.9, 512 / 256 9.2 / 8.3; K 11, C 128, 372 / 192 8.8 / 8.1;
// ups.0, 256 / 128 10.1 / 11.9, 576 / 288 19.5 / 18.5; conv_post 342 / 171 7.1 / 6.8, 744 / 384
// 9.7 / 9.8.  Grouped launches, whose problems are of different weight, from 200 (per depth of an
// MRF-256 stack, 384 / 192 10.8 / 11.8, 696 / 360 16.0 / 14.5).
static void choose_tiles(const ptk_conv_desc *const *ds, int n, int *S_out, int *nb_out) {
  const int env_s = knob(KN_CONV_SPLIT), env_nb = knob(KN_CONV_NB);
  bool nb2_ok = true;
  long long wgs1 = 0, wgs = 0, item = 0;
  for (int i = 0; i < n; i++) {
    const ptk_conv_desc *d = ds[i];
    if (conv_window(d, 2) > 32 * CONV_NU_MAX) nb2_ok = false;
    const long long mt = (d->M + 31) / 32, nq = d->nq_shape > 0 ? d->nq_shape : d->nq;
    wgs1 += d->batch * mt * ((d->nq + 31) / 32);
    wgs += d->batch * mt * ((d->nq + 63) / 64);
    item += mt * ((nq + 63) / 64);
  }
  const bool two = n > 1 ? wgs >= 200 : wgs >= 512 || (wgs + 255) / 256 < (wgs1 + 255) / 256;
  *nb_out = nb2_ok && (env_nb == 2 || (env_nb != 1 && two)) ? 2 : 1;
  *S_out = env_s == 2 || env_s == 4 ? env_s : item >= 640 ? 2 : 4;
}

// Order of three grouped problems (given heaviest first).  Workgroups are handed round the CUs in
// order, so in a launch that is resident at once the last problem's land on the CUs the first one's
// went to.  Heaviest first is right once CUs take several rounds; below that the heaviest belongs
// second, so that the lightest joins the middle one (per depth at C 256, T 904: 33.1 -> 31.3 us,
// T 720: 31.8 -> 28.5), and with two-wave workgroups, a problem of up to one per CU, last but the
// lightest second (C 128, T 3616: 35.1 -> 33.1 us, T 3472: 35.1 -> 32.6).
static void order_problems(const ptk_conv_desc **ds, int n, int S, int nb) {
  if (n != 3) return;
  long long total = 0, most = 0;
  for (int i = 0; i < 3; i++) {
    const long long wgs = (long long) ds[i]->batch * ((ds[i]->M + 31) / 32) * ((ds[i]->nq + 32 * nb - 1) / (32 * nb));
    total += wgs;
    if (wgs > most) most = wgs;
  }
  const int cus = 256;
  if (total > 12 / S * cus) return;   // more than are resident at once (three waves per SIMD)
  const int a = S == 2 && most <= cus ? 1 : 0;   // swap the last two, or the first two
  const ptk_conv_desc *t = ds[a];
  ds[a] = ds[a + 1];
  ds[a + 1] = t;
}

extern "C" int ptk_conv_mfma_ok(const ptk_conv_desc *d) {
  if (d->M < 16 || d->cin < 2 || d->K < 1 || d->stride < 1 || d->dil == 0) return 0;
  if (conv_window(d, 1) > 32 * CONV_NU_MAX) return 0;
  if (d->cinp != ptk_conv_cinp(d->cin)) return 0;
  // 32-bit buffer offsets: every row offset plus the out-of-range marker must stay below 2^32
  if ((unsigned long long) d->cinp * (unsigned long long) d->ldx * 4ULL >= 0x80000000ULL) return 0;
  return 1;
}

extern "C" int ptk_conv_stats(uint64_t out[2]) {
  HCHK(hipDeviceSynchronize());
  HCHK(hipMemcpyFromSymbol(out, HIP_SYMBOL(conv_stat), 2 * sizeof(uint64_t)));
  return 0;
}

template <int KT, int NB, int IN>
static void launch_conv_s(int S, const ConvGroup &g, dim3 grid, hipStream_t s) {
  const size_t lds = ((size_t) S * g.wslots + CONV_EXTRA_SLOTS) * 16;
#define CONV_LAUNCH(SV) \
  hipLaunchKernelGGL((conv_mfma_kernel<KT, NB, IN, SV>), grid, dim3(64 * SV), lds, s, g)
  if (S == 4) CONV_LAUNCH(4);
  else CONV_LAUNCH(2);
#undef CONV_LAUNCH
}
template <int KT, int NB>
static void launch_conv_in(int in_op, int S, const ConvGroup &g, dim3 grid, hipStream_t s) {
  if (in_op == PTK_IN_SPLIT) return launch_conv_s<KT, NB, PTK_IN_SPLIT>(S, g, grid, s);
  if (in_op == PTK_IN_LEAKY) launch_conv_s<KT, NB, PTK_IN_LEAKY>(S, g, grid, s);
  else launch_conv_s<KT, NB, PTK_IN_PLAIN>(S, g, grid, s);
}

extern "C" int ptk_conv_launch(const ptk_conv_desc *dd, int ngroup, void *stream) {
  if (ngroup < 1 || ngroup > PTK_MAX_GROUP) {
    set_err("ptk_conv_launch: ngroup %d out of range", ngroup);
    return -1;
  }
  ConvGroup g;
  memset(&g, 0, sizeof g);
  // heaviest problems first, so their long workgroups start before the short ones
  int order[PTK_MAX_GROUP];
  for (int i = 0; i < ngroup; i++) order[i] = i;
  for (int i = 0; i < ngroup; i++)
    for (int j = i + 1; j < ngroup; j++)
      if ((long long) dd[order[j]].K * dd[order[j]].cinp > (long long) dd[order[i]].K * dd[order[i]].cinp) {
        const int t = order[i];
        order[i] = order[j];
        order[j] = t;
      }
  int in_op = -1;
  int total = 0;
  const ptk_conv_desc *live[PTK_MAX_GROUP];
  for (int i = 0; i < ngroup; i++) {
    const ptk_conv_desc *d = &dd[order[i]];
    if (!ptk_conv_mfma_ok(d)) {
      set_err("ptk_conv_launch: shape outside the MFMA kernel (M %d cin %d K %d dil %d stride %d)",
              d->M, d->cin, d->K, d->dil, d->stride);
      return -1;
    }
    if (d->nq <= 0 || d->batch <= 0) continue;
    if (d->ext_l < 0 || d->ext_r < 0 || d->nq_shape < 0 || d->ext_l >= (1LL << 30) ||
        d->ext_r >= (1LL << 30)) {
      set_err("ptk_conv_launch: column extension or shape width out of range");
      return -1;
    }
    // a row tile's weight panel is addressed through one buffer resource (the input rows are
    // bounded the same way by ptk_conv_mfma_ok)
    if ((unsigned long long) d->K * (unsigned long long) (d->cinp / CONV_CK) * CONV_TAPB >= (unsigned long long) PTK_OOB) {
      set_err("ptk_conv_launch: weight panel (K %d, cin %d) reaches the 2 GiB range of one buffer "
              "resource", d->K, d->cin);
      return -1;
    }
    if (d->phase_il && !(d->M == 4 * d->C4 && d->C4 % 8 == 0 && d->ys == 4 && d->dil == -1 && d->stride == 1 &&
                         d->K == 4 && ngroup == 1)) {
      set_err("ptk_conv_launch: rows interleaved by phase need a single stride-4 convT in the "
              "4-tap phase form (M %d, rows per phase %d, %d taps)", d->M, d->C4, d->K);
      return -1;
    }
    if (d->in_op != PTK_IN_PLAIN && !(d->in_a >= 0.0f && d->in_a <= 1.0f)) {
      set_err("ptk_conv_launch: input LeakyReLU slope %g outside [0, 1]", (double) d->in_a);
      return -1;
    }
    if (in_op < 0) in_op = d->in_op;
    if (d->in_op == PTK_IN_SPLIT && (d->xsp == nullptr || d->cin % 16 != 0 || d->bsx % 4 != 0 ||
                                     ((uintptr_t) d->xsp & 15) != 0)) {
      set_err("ptk_conv_launch: split planes need channels in multiples of 16 and 16-byte columns");
      return -1;
    }
    if (d->ysp != nullptr && (d->C4 % 8 != 0 || d->bsy % 4 != 0 || ((uintptr_t) d->ysp & 15) != 0)) {
      set_err("ptk_conv_launch: a split output needs channels in multiples of 8 and 16-byte columns");
      return -1;
    }
    if (d->in_op != in_op || d->in_op < PTK_IN_PLAIN || d->in_op > PTK_IN_SPLIT) {
      set_err("ptk_conv_launch: grouped problems need one valid input transform");
      return -1;
    }
    live[g.ngroup] = d;
    g.ngroup++;
  }
  if (g.ngroup == 0) return 0;
  int maxcount = 0, S, nb, nu = 0;
  choose_tiles(live, g.ngroup, &S, &nb);
  order_problems(live, g.ngroup, S, nb);
  for (int i = 0; i < g.ngroup; i++) {
    const ptk_conv_desc *d = live[i];
    g.d[i] = *d;
    ConvProb &pi = g.info[i];
    const long long cols = 32LL * nb;   // columns of one tile
    const bool straight = d->stride == 1 && d->cin == d->cinp &&
                          (d->K == 4 ? g.ngroup == 1 : d->K == 3 || d->K == 7 || d->K == 11);
    const int need = straight && conv_window(d, nb) <= 32 * (nb + 1) ? nb + 1 : CONV_NU_MAX;
    if (need > nu) nu = need;
    pi.mt = (d->M + 31) / 32;
    const long long nt = (d->nq + cols - 1) / cols;
    long long nt0 = (d->nq + d->ext_l + cols - 1) / cols, n;
    if (d->batch == 1) {
      nt0 = (d->nq + d->ext_l + d->ext_r + cols - 1) / cols;
      n = pi.mt * nt0;
    } else {
      n = pi.mt * (nt0 + (d->batch - 2) * nt + (d->nq + d->ext_r + cols - 1) / cols);
    }
    if (n >= (1LL << 24) || total + n >= (1LL << 31)) {
      set_err("ptk_conv_launch: %lld workgroups for one problem (the tile decode takes < 2^24)", n);
      return -1;
    }
    // 32-bit columns: with fewer than 2^24 workgroups a column index times the stride stays below
    // 2^31 for every window the kernel takes unless the range itself starts far out
    const int kd = (d->K - 1) * d->dil;
    if ((d->q0 + d->nq + d->ext_r + 64) * d->stride + (kd < 0 ? -kd : kd) >= (1LL << 31) ||
        (d->q0 - d->ext_l) * d->stride + (kd < 0 ? kd : 0) - d->shift < -(1LL << 31) || d->lim >= (1LL << 31)) {
      set_err("ptk_conv_launch: columns past 2^31 (q0 %lld, nq %lld, stride %d)", (long long) d->q0,
              (long long) d->nq, d->stride);
      return -1;
    }
    total += (int) n;
    pi.count = (int) n;
    if (pi.count > maxcount) maxcount = pi.count;
    pi.mtnt = (int) (pi.mt * nt);
    pi.mtnt0 = (int) (pi.mt * nt0);
    pi.last = d->batch - 1;
    pi.div_tiles = fast_div((unsigned) pi.mtnt);
    pi.div_mt = fast_div((unsigned) pi.mt);
    const bool il = d->phase_il != 0;
    const bool one_phase = !il && (d->C4 == d->M || d->C4 % 32 == 0);
    if (one_phase && d->C4 != d->M) pi.div_phase = fast_div((unsigned) (d->C4 / 32));   // else m = 0: 0
    pi.q0 = (int) d->q0;
    pi.x = d->in_op == PTK_IN_SPLIT ? d->xsp : (const void *) d->x;
    pi.w = d->w;
    pi.scale = d->w + 2ll * (pi.mt * 32) * d->K * d->cinp;
    pi.bias = d->bias;
    pi.nbias4 = d->bias ? (int) (4 * (d->nbias < d->M ? d->nbias : d->M)) : 0;
    pi.C4 = d->C4;
    pi.K = d->K;
    pi.dil = d->dil;
    pi.st = d->stride;
    pi.cin = d->cin;
    pi.nchunk = d->cinp / CONV_CK;
    pi.ldx4 = (int) (d->ldx * 4);
    pi.lim = (int) d->lim;
    pi.shift = d->shift;
    pi.bsx = d->bsx;
    pi.kd = kd;
    pi.xw = conv_window(d, nb);
    pi.in_a = d->in_a;
    pi.addt = -1;
    int naddt = 0;
    for (int e = 0; e < d->nepi; e++)
      if (d->epi[e].op == PTK_EPI_ADDT && naddt++ == 0) pi.addt = e;
    pi.M = d->M;
    // the fast epilogue's 32-bit indices: columns, and byte offsets from a row block's first row
    const long long lim31 = 1LL << 31, lim30 = 1LL << 30;
    bool fast = (one_phase || il) && d->ldy < (1LL << 23) && d->Lout < lim30 &&
                (d->q0 + d->nq + d->ext_r) * d->ys + d->C4 < lim30 && d->q0 - d->ext_l >= 0 &&
                (32 * d->ldy + d->Lout) * 4 < lim31;
    // the fast epilogue reads one tensor operand (loaded ahead of the reduction); a chain with two
    // takes the general path
    if (naddt > 1) fast = false;
    // the interleaved-phase stores have no tensor-add operand loads: such a chain takes the
    // general path
    if (il && pi.addt >= 0) fast = false;
    // PTK_CONV_FAST=0: every block through the general per-element epilogue (tests compare the
    // two epilogues)
    if (!knob(KN_CONV_FAST)) fast = false;
    if (pi.addt >= 0) {
      const long long ldt = d->epi[pi.addt].ldt;
      fast = fast && ldt >= 0 && ldt < (1LL << 23) && (32 * ldt + d->Lout) * 4 < lim31;
    }
    pi.flags = (one_phase ? PROB_ONE_PHASE : 0) | (fast ? PROB_FAST : 0) | (il ? PROB_PHASE_IL : 0) |
               (d->reflect_l1 ? PROB_REFLECT : 0);
    pi.ext_l = (int) d->ext_l;
    pi.qend = (int) (d->q0 + d->nq);
    pi.ext_r = (int) d->ext_r;
    ConvEpi &ep = g.ep[i];
    ep.y = d->y;
    ep.y2 = d->y2;
    ep.ysp = d->ysp;
    ep.bsy = d->bsy;
    ep.t = pi.addt >= 0 ? d->epi[pi.addt].t : nullptr;
    ep.bst = pi.addt >= 0 ? d->epi[pi.addt].bst : 0;
    ep.ldy = (int) d->ldy;
    ep.ldt = pi.addt >= 0 ? (int) d->epi[pi.addt].ldt : 0;
    ep.lout = (int) d->Lout;
    ep.qend = (int) (d->q0 + d->nq);
    ep.ext_r = (int) d->ext_r;
    ep.ys = d->ys;
    ep.ypad = d->ypad;
    ep.C4 = d->C4;
    ep.nepi = d->nepi;
    ep.ops = 0;
    for (int e = 0; e < PTK_MAX_EPI; e++) {
      const int op = e < d->nepi ? d->epi[e].op : PTK_EPI_NONE;
      // codes outside the table are no-ops, as in epi_apply
      ep.ops |= (op >= PTK_EPI_NONE && op <= PTK_EPI_DIVS ? op : PTK_EPI_NONE) << (4 * e);
      ep.a[e] = e < d->nepi ? d->epi[e].a : 0.0f;
    }
    ep.a2 = d->a2;
  }
  if (total == 0) return 0;
  hipStream_t s = (hipStream_t) stream;
  const dim3 grid((unsigned) maxcount, (unsigned) g.ngroup);
  g.wslots = conv_slots(nu, nb);
  for (int i = 0; i < g.ngroup; i++) g.info[i].wslots = g.wslots;
  g.wcols = 32 * nu;
  const bool k4 = g.ngroup == 1 && g.d[0].K == 4;
  if (nb == 2 && k4) launch_conv_in<4, 2>(in_op, S, g, grid, s);
  else if (nb == 2) launch_conv_in<11, 2>(in_op, S, g, grid, s);
  else if (k4) launch_conv_in<4, 1>(in_op, S, g, grid, s);
  else launch_conv_in<11, 1>(in_op, S, g, grid, s);
  HCHK(hipGetLastError());
  return 0;
}

// ------------------------------------------------------------------------------ narrow convs
// Convs and convTs with few output rows on the reference ABI path (cout4 < 16, channel counts 1,
// 4 or 16: the PQMF synthesis FIR 4 -> 1 K 63; the iSTFT overlap-add 16 -> 1 and window sum
// 1 -> 1, K 16 s 4; the PQMF x4 zero-insert 4 -> 4 K 4 s 4).  A workgroup stages in LDS, once,
// the input window its outputs read, as [column][CIN] (a column's channels in one to four 16-byte
// reads; the column stride padded to CIN + 4 floats for CIN 16, so a wave's reads spread over all
// banks), and the real rows' weights, [row][tap][CIN] (conv) or [row][tap][CIN][s] (convT).  Each
// output is one chain of FMAs in the generic kernels' order (bias, tap ascending, channel
// ascending, taps whose input column is outside the sequence skipped), so the results are the
// same bits.  The chip is nearly empty at these sizes, so the work is spread over many waves: one
// conv output per thread, its taps' operands read one tap ahead into two alternating register
// sets; a convT step's s phases per thread, sharing each input value.  (A first form, a plain loop
// with its reads waiting one at a time, took 14-38 us per launch; four conv outputs per thread
// gave 228 waves each issuing ~4700 instructions one at a time: 19 us.)  The layout's padding rows
// (cout..cout4-1, zero weights and bias) get the epilogue of 0 without the sums.  Other channel
// counts, windows past NARROW_LDS_FLOATS and sizes past 2^31 take the generic kernels below;
// PTK_NARROW=0 forces them everywhere.
#define NARROW_THREADS 256
#define NARROW_LDS_FLOATS 12288   // 48 KB of dynamic LDS per workgroup
#define NARROW_SMAX 4             // convT phases (stride) a thread keeps in registers

// floats per staged window column
template <int CIN>
__host__ __device__ constexpr int narrow_cs() { return CIN >= 16 ? CIN + 4 : CIN; }

// CIN consecutive floats from LDS (16-byte aligned when CIN % 4 == 0) into registers
template <int CIN>
__device__ __forceinline__ void lds_cols(float (&v)[CIN], const float *p) {
  if constexpr (CIN % 4 == 0) {
#pragma unroll
    for (int q = 0; q < CIN / 4; q++) {
      const float4 t = reinterpret_cast<const float4 *>(p)[q];
      v[4 * q] = t.x;
      v[4 * q + 1] = t.y;
      v[4 * q + 2] = t.z;
      v[4 * q + 3] = t.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < CIN; i++) v[i] = p[i];
  }
}

// Stages columns [0, win) of rows [0, CIN) into xs[col][narrow_cs<CIN>] (column c0 + col of the
// item, 0 outside [0, lim)).  A thread's columns col = tid + p * NARROW_THREADS are taken PG at a
// time, and all PG * CIN loads of a group are issued before its stores, so the window costs about
// one global load latency per group.
template <int CIN>
__device__ __forceinline__ void narrow_stage(float *__restrict__ xs, const float *__restrict__ xb,
                                             long long ldx, int c0, int lim, int win, int tid) {
  constexpr int PG = CIN >= 16 ? 2 : 16 / CIN, CS = narrow_cs<CIN>();
  for (int col0 = tid; col0 < win; col0 += PG * NARROW_THREADS) {
    float v[PG][CIN];
#pragma unroll
    for (int g = 0; g < PG; g++) {
      const int c = c0 + col0 + g * NARROW_THREADS;
      const bool ok = col0 + g * NARROW_THREADS < win && c >= 0 && c < lim;
      const float *src = xb + (ok ? c : 0);
#pragma unroll
      for (int ci = 0; ci < CIN; ci++) v[g][ci] = ok ? src[(long long) ci * ldx] : 0.0f;
    }
#pragma unroll
    for (int g = 0; g < PG; g++) {
      const int col = col0 + g * NARROW_THREADS;
      if (col >= win) break;
      if constexpr (CIN % 4 == 0) {
#pragma unroll
        for (int q = 0; q < CIN / 4; q++)
          reinterpret_cast<float4 *>(xs + col * CS)[q] =
              make_float4(v[g][4 * q], v[g][4 * q + 1], v[g][4 * q + 2], v[g][4 * q + 3]);
      } else {
#pragma unroll
        for (int ci = 0; ci < CIN; ci++) xs[col * CS + ci] = v[g][ci];
      }
    }
  }
}

template <int CIN>
__device__ __forceinline__ float narrow_fma(float acc, const float (&w)[CIN], const float (&x)[CIN]) {
#pragma unroll
  for (int ci = 0; ci < CIN; ci++) acc += w[ci] * x[ci];
  return acc;
}

template <int CIN>
__global__ void __launch_bounds__(NARROW_THREADS) conv_narrow_kernel(
    const float *__restrict__ x, long long ldx, long long bsx, int lim, const float *__restrict__ wp,
    const float *__restrict__ bias, int cout, int K, int st, int dil, int shift,
    float *__restrict__ y, long long ldy, long long bsy, int n, int win, int epi0, float a0,
    int epi1, float a1) {
  constexpr int CS = narrow_cs<CIN>();
  extern __shared__ float4 lds4[];
  float *const xs = reinterpret_cast<float *>(lds4);   // [win][CS]; column 0 = input t0*st - shift
  float *const ws = xs + ((win * CS + 3) & ~3);        // [cout][K][CIN]
  const int tid = threadIdx.x, b = blockIdx.y;
  const int t0 = blockIdx.x * NARROW_THREADS;
  narrow_stage<CIN>(xs, x + (long long) b * bsx, ldx, t0 * st - shift, lim, win, tid);
  for (int i = tid; i < cout * K * CIN; i += NARROW_THREADS) {
    const int m = i / (K * CIN), r = i - m * (K * CIN), k = r / CIN, ci = r - k * CIN;
    ws[i] = wp[((long long) (m >> 2) * K + k) * CIN * 4 + ci * 4 + (m & 3)];
  }
  __syncthreads();
  const int t = t0 + tid;
  if (t >= n) return;
  // taps whose input column t * st + k * dil - shift lies in [0, lim): k in [klo, khi)
  const int base = t * st - shift;
  int klo = base >= 0 ? 0 : (-base + dil - 1) / dil;
  int khi = base >= lim ? 0 : (lim - base + dil - 1) / dil;
  khi = khi < K ? khi : K;
  klo = klo < khi ? klo : khi;
  const int c4 = (cout + 3) & ~3;
  const ptk_epi e0 = {epi0, a0, nullptr, 0, 0}, e1 = {epi1, a1, nullptr, 0, 0};
  const float *const xt = xs + tid * st * CS;
  const int kstep = dil * CS;
  for (int m = 0; m < c4; m++) {
    float v = (bias != nullptr && m < cout) ? bias[m] : 0.0f;
    if (m < cout && klo < khi) {
      const float *const wm = ws + m * K * CIN;
      // operands of the next tap read into the other register set while this tap's FMAs run;
      // the read is unconditional (a tap past the last re-reads the last), so the wait before
      // the FMAs leaves it in flight
      const int klast = khi - 1;
      float wa[CIN], xa[CIN], wb[CIN], xb2[CIN];
      lds_cols<CIN>(wa, wm + klo * CIN);
      lds_cols<CIN>(xa, xt + klo * kstep);
      for (int k = klo;; k += 2) {
        const int k1 = k + 1 < klast ? k + 1 : klast, k2 = k + 2 < klast ? k + 2 : klast;
        lds_cols<CIN>(wb, wm + k1 * CIN);
        lds_cols<CIN>(xb2, xt + k1 * kstep);
        v = narrow_fma<CIN>(v, wa, xa);
        if (k + 1 >= khi) break;
        lds_cols<CIN>(wa, wm + k2 * CIN);
        lds_cols<CIN>(xa, xt + k2 * kstep);
        v = narrow_fma<CIN>(v, wb, xb2);
        if (k + 2 >= khi) break;
      }
    }
    if (epi0) v = epi_apply(v, e0, b, m, t);
    if (epi1) v = epi_apply(v, e1, b, m, t);
    y[(long long) b * bsy + (long long) m * ldy + t] = v;
  }
}

// Thread tid of workgroup bx takes the delay-line step q = qlo + bx * NARROW_THREADS + tid and its
// s outputs oi = q * s + r - pad (r < s) that fall in [0, Lout), all s phases at once (s
// independent sums over the same input values); the window holds input columns
// [q0 - ntap + 1, q0 + NARROW_THREADS) of the workgroup's first step q0.
template <int CIN>
__global__ void __launch_bounds__(NARROW_THREADS) convT_narrow_kernel(
    const float *__restrict__ x, long long ldx, long long bsx, int tin, const float *__restrict__ wp,
    const float *__restrict__ bias, int cout, int s, int pad, int ntap, float *__restrict__ y,
    long long ldy, long long bsy, int Lout, int qlo, int nq, int win) {
  constexpr int CS = narrow_cs<CIN>();
  extern __shared__ float4 lds4[];
  float *const xs = reinterpret_cast<float *>(lds4);   // [win][CS]
  float *const ws = xs + ((win * CS + 3) & ~3);        // [cout][ntap][CIN][NARROW_SMAX]
  const int tid = threadIdx.x, b = blockIdx.y;
  const int c4 = (cout + 3) & ~3;
  const int q0 = qlo + blockIdx.x * NARROW_THREADS;
  narrow_stage<CIN>(xs, x + (long long) b * bsx, ldx, q0 - ntap + 1, tin, win, tid);
  for (int i = tid; i < cout * ntap * CIN * NARROW_SMAX; i += NARROW_THREADS) {
    const int r = i % NARROW_SMAX, rest = i / NARROW_SMAX, ci = rest % CIN, rest2 = rest / CIN;
    const int j = rest2 % ntap, co = rest2 / ntap, row = r * c4 + co;
    ws[i] = r < s ? wp[((long long) (row >> 2) * ntap + j) * CIN * 4 + ci * 4 + (row & 3)] : 0.0f;
  }
  __syncthreads();
  const int q = q0 + tid;
  if (q - qlo >= nq) return;
  // taps whose input column q - j lies in [0, tin): j in [jlo, jhi)
  const int jlo = q >= tin ? q - tin + 1 : 0;
  const int jhi = q + 1 < ntap ? q + 1 : ntap;
  float *yb = y + (long long) b * bsy;
  const float *const xq = xs + (tid + ntap - 1) * CS;   // input column q - j at xq[-j * CS]
  for (int co = 0; co < c4; co++) {
    const float bv = (bias != nullptr && co < cout) ? bias[co] : 0.0f;
    float acc[NARROW_SMAX];
#pragma unroll
    for (int r = 0; r < NARROW_SMAX; r++) acc[r] = bv;
    if (co < cout) {
      const float *const wc = ws + co * ntap * CIN * NARROW_SMAX;
      for (int j = jlo; j < jhi; j++) {
        // the tap's operands all read before its FMAs
        float xv[CIN], w[CIN][NARROW_SMAX];
        lds_cols<CIN>(xv, xq - j * CS);
#pragma unroll
        for (int ci = 0; ci < CIN; ci++) lds_cols<NARROW_SMAX>(w[ci], wc + (j * CIN + ci) * NARROW_SMAX);
#pragma unroll
        for (int ci = 0; ci < CIN; ci++)
#pragma unroll
          for (int r = 0; r < NARROW_SMAX; r++) acc[r] += w[ci][r] * xv[ci];
      }
    }
#pragma unroll
    for (int r = 0; r < NARROW_SMAX; r++) {
      const int oi = q * s + r - pad;
      if (r < s && oi >= 0 && oi < Lout) yb[(long long) co * ldy + oi] = acc[r];
    }
  }
}

// ------------------------------------------------------------------------------ SIMT fallbacks
// Any shape the MFMA and narrow kernels do not take: one thread per output, summing over tap then
// channel onto the bias in the reference's order.
__global__ void conv_simt_kernel(const float *__restrict__ x, long long ldx, long long bsx,
                                 long long lim, int cin, const float *__restrict__ wp,
                                 const float *__restrict__ bias, int cout, int K, int st, int dil,
                                 int shift, float *__restrict__ y, long long ldy, long long bsy,
                                 long long n, int epi0, float a0, int epi1, float a1) {
  const long long t = (long long) blockIdx.x * blockDim.x + threadIdx.x;
  const int m = blockIdx.y, b = blockIdx.z;
  if (t >= n) return;
  const float *xb = x + (long long) b * bsx;
  const float *wq = wp + (long long) (m >> 2) * K * cin * 4 + (m & 3);
  float v = (bias != nullptr && m < cout) ? bias[m] : 0.0f;
  for (int k = 0; k < K; k++) {
    const long long c = t * st + (long long) k * dil - shift;
    if (c < 0 || c >= lim) continue;
    const float *wk = wq + (long long) k * cin * 4;
    for (int ci = 0; ci < cin; ci++) v += wk[ci * 4] * xb[(long long) ci * ldx + c];
  }
  ptk_epi e0 = {epi0, a0, nullptr, 0, 0}, e1 = {epi1, a1, nullptr, 0, 0};
  if (epi0) v = epi_apply(v, e0, b, m, t);
  if (epi1) v = epi_apply(v, e1, b, m, t);
  y[(long long) b * bsy + (long long) m * ldy + t] = v;
}

extern "C" int ptk_conv_simt(const float *x, int64_t ldx, int64_t bsx, int64_t lim, int cin,
                             const float *wp, const float *bias, int cout, int K, int stride,
                             int dil, int shift, float *y, int64_t ldy, int64_t bsy, int64_t n,
                             int batch, int epi0, float a0, int epi1, float a1, void *s) {
  if (n <= 0 || batch <= 0) return 0;
  // no residual tensor reaches these kernels: a tensor add would read through a null pointer
  if (epi0 == PTK_EPI_ADDT || epi1 == PTK_EPI_ADDT) {
    set_err("ptk_conv_simt: epilogue code %d (tensor add) takes no tensor here", PTK_EPI_ADDT);
    return -1;
  }
  const long long per_wg = NARROW_THREADS;
  const long long win = (per_wg - 1) * stride + (long long) (K - 1) * dil + 1;
  const long long cs = cin >= 16 ? cin + 4 : cin;
  const long long lds_floats = ((cs * win + 3) & ~3LL) + (long long) cout * K * cin;
  // 32-bit column arithmetic in the kernel: every window column, output and input index < 2^31
  const bool small = lim < INT32_MAX && (n + per_wg) * stride + win + shift < INT32_MAX;
  if (knob(KN_NARROW) && (cin == 1 || cin == 4 || cin == 16) && dil >= 1 && stride >= 1 && small &&
      lds_floats <= NARROW_LDS_FLOATS) {
    dim3 grid((unsigned) ((n + per_wg - 1) / per_wg), (unsigned) batch);
    const size_t lds = (size_t) lds_floats * sizeof(float);
#define NARROW_CONV_LAUNCH(CINV)                                                                  \
  hipLaunchKernelGGL(conv_narrow_kernel<CINV>, grid, dim3(NARROW_THREADS), lds, (hipStream_t) s, x, \
                     (long long) ldx, (long long) bsx, (int) lim, wp, bias, cout, K, stride, dil,  \
                     shift, y, (long long) ldy, (long long) bsy, (int) n, (int) win, epi0, a0,     \
                     epi1, a1)
    if (cin == 1) NARROW_CONV_LAUNCH(1);
    else if (cin == 4) NARROW_CONV_LAUNCH(4);
    else NARROW_CONV_LAUNCH(16);
#undef NARROW_CONV_LAUNCH
    HCHK(hipGetLastError());
    return 0;
  }
  const int c4 = (cout + 3) / 4 * 4;
  dim3 grid((unsigned) ((n + 255) / 256), (unsigned) c4, (unsigned) batch);
  hipLaunchKernelGGL(conv_simt_kernel, grid, dim3(256), 0, (hipStream_t) s, x, (long long) ldx,
                     (long long) bsx, (long long) lim, cin, wp, bias, cout, K, stride, dil, shift,
                     y, (long long) ldy, (long long) bsy, (long long) n, epi0, a0, epi1, a1);
  HCHK(hipGetLastError());
  return 0;
}

__global__ void convT_simt_kernel(const float *__restrict__ x, long long ldx, long long bsx,
                                  long long tin, int cin, const float *__restrict__ wp,
                                  const float *__restrict__ bias, int cout, int s, int pad, int ntap,
                                  float *__restrict__ y, long long ldy, long long bsy, long long Lout) {
  const long long oi = (long long) blockIdx.x * blockDim.x + threadIdx.x;
  const int co = blockIdx.y, b = blockIdx.z;
  if (oi >= Lout) return;
  const int c4 = (cout + 3) / 4 * 4;
  const long long u = oi + pad;
  const long long q = u / s;
  const int r = (int) (u - q * s);
  const int row = r * c4 + co;
  const float *wq = wp + (long long) (row >> 2) * ntap * cin * 4 + (row & 3);
  const float *xb = x + (long long) b * bsx;
  float v = (bias != nullptr && co < cout) ? bias[co] : 0.0f;
  for (int j = 0; j < ntap; j++) {
    const long long c = q - j;
    if (c < 0 || c >= tin) continue;
    const float *wj = wq + (long long) j * cin * 4;
    for (int ci = 0; ci < cin; ci++) v += wj[ci * 4] * xb[(long long) ci * ldx + c];
  }
  y[(long long) b * bsy + (long long) co * ldy + oi] = v;
}

extern "C" int ptk_convT_simt(const float *x, int64_t ldx, int64_t bsx, int64_t tin, int cin,
                              const float *wp, const float *bias, int cout, int st, int pad, int K,
                              float *y, int64_t ldy, int64_t bsy, int64_t Lout, int batch, void *s) {
  if (Lout <= 0 || batch <= 0) return 0;
  const int c4 = (cout + 3) / 4 * 4;
  const int ntap = (K + st - 1) / st;
  const long long win = NARROW_THREADS + ntap - 1;
  const long long cs = cin >= 16 ? cin + 4 : cin;
  const long long lds_floats = ((cs * win + 3) & ~3LL) + (long long) NARROW_SMAX * cout * ntap * cin;
  const bool small = tin < INT32_MAX - NARROW_THREADS && Lout + pad + (long long) NARROW_THREADS * st < INT32_MAX;
  if (knob(KN_NARROW) && (cin == 1 || cin == 4 || cin == 16) && st >= 1 && st <= NARROW_SMAX &&
      pad >= 0 && small && lds_floats <= NARROW_LDS_FLOATS) {
    // delay-line steps with an output in [0, Lout): u = oi + pad = q * st + r
    const long long qlo = pad / st, nq = (Lout - 1 + pad) / st - qlo + 1;
    dim3 grid((unsigned) ((nq + NARROW_THREADS - 1) / NARROW_THREADS), (unsigned) batch);
    const size_t lds = (size_t) lds_floats * sizeof(float);
#define NARROW_CONVT_LAUNCH(CINV)                                                                 \
  hipLaunchKernelGGL(convT_narrow_kernel<CINV>, grid, dim3(NARROW_THREADS), lds, (hipStream_t) s, \
                     x, (long long) ldx, (long long) bsx, (int) tin, wp, bias, cout, st, pad, ntap, \
                     y, (long long) ldy, (long long) bsy, (int) Lout, (int) qlo, (int) nq, (int) win)
    if (cin == 1) NARROW_CONVT_LAUNCH(1);
    else if (cin == 4) NARROW_CONVT_LAUNCH(4);
    else NARROW_CONVT_LAUNCH(16);
#undef NARROW_CONVT_LAUNCH
    HCHK(hipGetLastError());
    return 0;
  }
  dim3 grid((unsigned) ((Lout + 255) / 256), (unsigned) c4, (unsigned) batch);
  hipLaunchKernelGGL(convT_simt_kernel, grid, dim3(256), 0, (hipStream_t) s, x, (long long) ldx,
                     (long long) bsx, (long long) tin, cin, wp, bias, cout, st, pad, ntap, y,
                     (long long) ldy, (long long) bsy, (long long) Lout);
  HCHK(hipGetLastError());
  return 0;
}

// ------------------------------------------------------------------------------ matmul
// fp32 MFMA matmul, C[m][n] = A[m][k] . B[k][n], all row-major with leading dimensions lda, ldb,
// ldc (the reference's pt_v21_matmul contract).  A workgroup computes a 64x64 block of C, each of
// its four waves a 32x32 tile, walking k in steps of 8: lane (h, r) feeds A[row r][k0 + 2p + h]
// and B[k0 + 2p + h][column r] to the p-th of four v_mfma_f32_32x32x2_f32 (the operand layout of
// the conv kernel).  Loads outside the matrices read as 0, so any m, n, k works.
__global__ void __launch_bounds__(256) matmul_mfma_kernel(const float *__restrict__ A, long long m,
                                                          long long k, long long lda,
                                                          const float *__restrict__ B,
                                                          long long ldb, long long nn,
                                                          float *__restrict__ C, long long ldc) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int h = lane >> 5, l32 = lane & 31;
  const long long r0 = (long long) blockIdx.y * 64 + (w >> 1) * 32;
  const long long c0 = (long long) blockIdx.x * 64 + (w & 1) * 32;
  const long long ra = r0 + l32, cb = c0 + l32;
  const bool rok = ra < m, cok = cb < nn;
  const float *arow = A + (rok ? ra : 0) * lda;
  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; v++) acc[v] = 0.0f;
  for (long long k0 = 0; k0 < k; k0 += 8) {
    float av[4], bv[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const long long kk = k0 + 2 * q + h;
      const bool kok = kk < k;
      av[q] = (rok && kok) ? arow[kk] : 0.0f;
      bv[q] = (cok && kok) ? B[kk * ldb + cb] : 0.0f;
    }
#pragma unroll
    for (int q = 0; q < 4; q++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[q], bv[q], acc, 0, 0, 0);
  }
#pragma unroll
  for (int v = 0; v < 16; v++) {
    const long long row = r0 + 8 * (v >> 2) + 4 * h + (v & 3);
    if (row < m && cok) C[row * ldc + cb] = acc[v];
  }
}
extern "C" int ptk_matmul(const float *A, int64_t m, int64_t k, int64_t lda, const float *B,
                          int64_t ldb, int64_t nn, float *C, int64_t ldc, void *s) {
  if (m <= 0 || nn <= 0) return 0;
  const long long gy = (m + 63) / 64, gx = (nn + 63) / 64;
  if (gy > 65535 || gx > 0x7fffffffLL) {
    set_err("ptk_matmul: %lld x %lld outside the grid limits", (long long) m, (long long) nn);
    return -1;
  }
  hipLaunchKernelGGL(matmul_mfma_kernel, dim3((unsigned) gx, (unsigned) gy), dim3(256), 0,
                     (hipStream_t) s, A, (long long) m, (long long) k, (long long) lda, B,
                     (long long) ldb, (long long) nn, C, (long long) ldc);
  HCHK(hipGetLastError());
  return 0;
}

// ------------------------------------------------------------------------------ elementwise
__global__ void add_kernel(const float *__restrict__ a, const float *__restrict__ b,
                           float *__restrict__ y, long long n, int epi, float alpha) {
  long long i = (long long) blockIdx.x * blockDim.x + threadIdx.x;
  const long long st = (long long) gridDim.x * blockDim.x;
  for (; i < n; i += st) {
    float v = a[i] + b[i];
    if (epi == 1) v = v >= 0.0f ? v : alpha * v;
    y[i] = v;
  }
}
__global__ void leaky_kernel(const float *__restrict__ a, float *__restrict__ y, long long n,
                             float alpha) {
  long long i = (long long) blockIdx.x * blockDim.x + threadIdx.x;
  const long long st = (long long) gridDim.x * blockDim.x;
  for (; i < n; i += st) {
    const float v = a[i];
    y[i] = v >= 0.0f ? v : alpha * v;
  }
}
__global__ void avg3_leaky_kernel(const float *__restrict__ a, const float *__restrict__ b,
                                  const float *__restrict__ c, float *__restrict__ y, long long n,
                                  float alpha) {
  long long i = (long long) blockIdx.x * blockDim.x + threadIdx.x;
  const long long st = (long long) gridDim.x * blockDim.x;
  for (; i < n; i += st) {
    const float v = ((a[i] + b[i]) + c[i]) / 3.0f;
    y[i] = v >= 0.0f ? v : alpha * v;
  }
}
static bool al16(const void *p) { return ((uintptr_t) p & 15) == 0; }
// leaky(((a + b) + c) / 3) of [items][C][T] tensors, as fp32 and as split planes: a thread per column
// of eight channels.  Memory-bound (five tensors' worth of traffic).
// Bound by HBM: at batch 8, T 226 9.1 us (C 256) and 11.9 us (C 128); the fp32-only pass it replaced
// took 5.6 and 9.7 us, and the convs behind it then split their input per row block.
__global__ void __launch_bounds__(128) avg3_leaky_split_kernel(
    const float *__restrict__ a, const float *__restrict__ b, const float *__restrict__ c,
    float *__restrict__ y, u32x4 *__restrict__ ysp, long long ngroup, int T, float alpha) {
  const int t = blockIdx.x * 128 + threadIdx.x;
  if (t >= T) return;
  for (long long g = blockIdx.y; g < ngroup; g += gridDim.y) {   // eight-channel groups of all items
    const long long i0 = g * 8 * T + t;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const long long i = i0 + (long long) e * T;
      const float s = ((a[i] + b[i]) + c[i]) / 3.0f;
      v[e] = s >= 0.0f ? s : alpha * s;
    }
    u32x4 h, l;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      unsigned hh, ll;
      split_input(v[2 * e], v[2 * e + 1], hh, ll);
      h[e] = hh;
      l[e] = ll;
    }
#pragma unroll
    for (int e = 0; e < 8; e++) y[i0 + (long long) e * T] = v[e];
    ysp[g * 2 * T + t] = h;
    ysp[(g * 2 + 1) * T + t] = l;
  }
}
extern "C" int ptk_avg3_leaky_split(const float *a, const float *b, const float *c, float *y, void *ysp,
                                    int64_t rows, int64_t T, float alpha, void *s) {
  if (rows <= 0 || T <= 0) return 0;
  if (rows % 8 != 0 || T >= INT_MAX - 128 || !al16(ysp)) {
    set_err("ptk_avg3_leaky_split: %lld rows of %lld columns", (long long) rows, (long long) T);
    return -1;
  }
  hipLaunchKernelGGL(avg3_leaky_split_kernel, dim3((unsigned) ((T + 127) / 128), (unsigned) (rows / 8 < 65535 ? rows / 8 : 65535)),
                     dim3(128), 0, (hipStream_t) s, a, b, c, y, reinterpret_cast<u32x4 *>(ysp),
                     (long long) (rows / 8), (int) T, alpha);
  HCHK(hipGetLastError());
  return 0;
}
static unsigned ew_blocks(long long n) {
  long long b = (n + 255) / 256;
  if (b > 8192) b = 8192;
  return (unsigned) (b < 1 ? 1 : b);
}

// The same elementwise ops four elements per thread, for 16-byte aligned operands (the decoder's
// arena blocks are 256-byte aligned): each element goes through exactly the scalar kernel's
// operations, the n % 4 tail elements through threads 0 .. n % 4 - 1.
__device__ __forceinline__ float leaky1(float v, float a) { return v >= 0.0f ? v : a * v; }
__global__ void avg3_leaky4_kernel(const float *__restrict__ a, const float *__restrict__ b,
                                   const float *__restrict__ c, float *__restrict__ y, long long n,
                                   float alpha) {
  const long long n4 = n >> 2, i0 = (long long) blockIdx.x * blockDim.x + threadIdx.x;
  const long long st = (long long) gridDim.x * blockDim.x;
  for (long long i = i0; i < n4; i += st) {
    const float4 va = reinterpret_cast<const float4 *>(a)[i], vb = reinterpret_cast<const float4 *>(b)[i],
                 vc = reinterpret_cast<const float4 *>(c)[i];
    reinterpret_cast<float4 *>(y)[i] = make_float4(leaky1(((va.x + vb.x) + vc.x) / 3.0f, alpha),
                                                   leaky1(((va.y + vb.y) + vc.y) / 3.0f, alpha),
                                                   leaky1(((va.z + vb.z) + vc.z) / 3.0f, alpha),
                                                   leaky1(((va.w + vb.w) + vc.w) / 3.0f, alpha));
  }
  if (i0 < (n & 3)) {
    const long long e = (n4 << 2) + i0;
    y[e] = leaky1(((a[e] + b[e]) + c[e]) / 3.0f, alpha);
  }
}
__global__ void add4_kernel(const float *__restrict__ a, const float *__restrict__ b,
                            float *__restrict__ y, long long n, int epi, float alpha) {
  const long long n4 = n >> 2, i0 = (long long) blockIdx.x * blockDim.x + threadIdx.x;
  const long long st = (long long) gridDim.x * blockDim.x;
  for (long long i = i0; i < n4; i += st) {
    const float4 va = reinterpret_cast<const float4 *>(a)[i], vb = reinterpret_cast<const float4 *>(b)[i];
    float4 v = make_float4(va.x + vb.x, va.y + vb.y, va.z + vb.z, va.w + vb.w);
    if (epi == 1) v = make_float4(leaky1(v.x, alpha), leaky1(v.y, alpha), leaky1(v.z, alpha), leaky1(v.w, alpha));
    reinterpret_cast<float4 *>(y)[i] = v;
  }
  if (i0 < (n & 3)) {
    const long long e = (n4 << 2) + i0;
    const float v = a[e] + b[e];
    y[e] = epi == 1 ? leaky1(v, alpha) : v;
  }
}
__global__ void leaky4_kernel(const float *__restrict__ a, float *__restrict__ y, long long n, float alpha) {
  const long long n4 = n >> 2, i0 = (long long) blockIdx.x * blockDim.x + threadIdx.x;
  const long long st = (long long) gridDim.x * blockDim.x;
  for (long long i = i0; i < n4; i += st) {
    const float4 va = reinterpret_cast<const float4 *>(a)[i];
    reinterpret_cast<float4 *>(y)[i] = make_float4(leaky1(va.x, alpha), leaky1(va.y, alpha),
                                                   leaky1(va.z, alpha), leaky1(va.w, alpha));
  }
  if (i0 < (n & 3)) y[(n4 << 2) + i0] = leaky1(a[(n4 << 2) + i0], alpha);
}
extern "C" int ptk_add(const float *a, const float *b, float *y, int64_t n, int epi, float alpha,
                       void *s) {
  if (n <= 0) return 0;
  if (al16(a) && al16(b) && al16(y) && n >= 4)
    hipLaunchKernelGGL(add4_kernel, dim3(ew_blocks(n >> 2)), dim3(256), 0, (hipStream_t) s, a, b, y,
                       (long long) n, epi, alpha);
  else
    hipLaunchKernelGGL(add_kernel, dim3(ew_blocks(n)), dim3(256), 0, (hipStream_t) s, a, b, y,
                       (long long) n, epi, alpha);
  HCHK(hipGetLastError());
  return 0;
}
extern "C" int ptk_avg3_leaky(const float *a, const float *b, const float *c, float *y, int64_t n,
                              float alpha, void *s) {
  if (n <= 0) return 0;
  if (al16(a) && al16(b) && al16(c) && al16(y) && n >= 4)
    hipLaunchKernelGGL(avg3_leaky4_kernel, dim3(ew_blocks(n >> 2)), dim3(256), 0, (hipStream_t) s, a,
                       b, c, y, (long long) n, alpha);
  else
    hipLaunchKernelGGL(avg3_leaky_kernel, dim3(ew_blocks(n)), dim3(256), 0, (hipStream_t) s, a, b,
                       c, y, (long long) n, alpha);
  HCHK(hipGetLastError());
  return 0;
}
extern "C" int ptk_leaky(const float *a, float *y, int64_t n, float alpha, void *s) {
  if (n <= 0) return 0;
  if (al16(a) && al16(y) && n >= 4)
    hipLaunchKernelGGL(leaky4_kernel, dim3(ew_blocks(n >> 2)), dim3(256), 0, (hipStream_t) s, a, y,
                       (long long) n, alpha);
  else
    hipLaunchKernelGGL(leaky_kernel, dim3(ew_blocks(n)), dim3(256), 0, (hipStream_t) s, a, y,
                       (long long) n, alpha);
  HCHK(hipGetLastError());
  return 0;
}

// ------------------------------------------------------------------------------ decoder tail
// conv_post output p [72][L] (channel c = band*18 + k) -> waveform, fused:
//   frame[b][n][t] = hann[n] * sum_k (re Bc[k][n] + im Bs[k][n]),  re/im = exp(p_k) cos/sin(pi sin(p_9+k))
//   ola[b][j] = sum_{j-4t in [0,16)} frame[b][j-4t][t];   y[b][i] = ola[b][i+8] / max(wsum[i+8], 1e-9)
//   wav[o] = sum_b sum_m h[b][m] * 4 * y[b][(o+m-31)/4]   over (o+m-31) = 0 mod 4 in range.
// A tile is TOUT consecutive samples of one item, made by one workgroup of four waves that
// recomputes the frames the tile needs, so the whole tail is a single pass over p with no
// intermediates in HBM.  Its two products run on the fp32 16x16x4 MFMA (lane l holds A[l%16][l/16],
// B[l/16][l%16] and result rows 4(l/16)+i of column l%16):
//   - the irfft: 16 frames x 16 samples per product group, the spectrum as A (k = the lane's bin
//     group: re of bin g, im of bin g (bin 0's k group carries re of bin 8 instead: the imaginary
//     parts of bins 0 and 8 meet sin(0) and sin(pi n), which vanish), re and im of bin g + 4), the
//     basis with hann folded in as B;
//   - the PQMF synthesis: samples o0' + 16m + 4q + r of a 256-sample block are
//     sum_b sum_s y_b[64k + 4m + 1 + s] * 4 h_b[3 - r + 4(s - q)], a Hankel product over the 19
//     shifts s with the four bands as the k of each MFMA.
// Wave w makes band w's frames and y values (phases A and B touch only that wave's LDS, so they
// need no barrier), then the waves make one 256-sample block each from all bands' y (phase C).
// A workgroup loops over tiles (tile, tile + gridDim.x, ...); the next tile's reads are issued as
// soon as the current tile's are used and arrive while phases B and C run.
// An angle p (radians) as revolutions in [-1/2, 1/2] for v_sin_f32 / v_cos_f32, whose input
// domain is |x| <= 256 revolutions and which see only the rounded product p / 2 pi.  Cody and
// Waite's two-constant reduction (W. J. Cody, W. Waite, Software Manual for the Elementary
// Functions, 1980): k = rint(p / 2 pi), r = (p - k C1) - k C2 with C1 = fp32(2 pi) and
// C2 = 2 pi - C1, each step one fused multiply-add, so r carries p's own bits to within a few
// units of its last place for |p| up to ~1e7.  For |p| < pi, k = 0 and r = p: the result is the
// plain p / 2 pi.
__device__ __forceinline__ float rev_of(float p) {
  const float k = __builtin_rintf(p * 0.159154943f);
  float r = __builtin_fmaf(-k, 6.28318548f, p);
  r = __builtin_fmaf(-k, -1.74845553e-7f, r);
  return r * 0.159154943f;
}

template <int TOUT>
struct TailGeo {
  static constexpr int NG = ((TOUT / 4 + 27) / 4 + 16) / 16;   // 16-frame groups per band
  static constexpr int P = 64 * NG + 32;     // one overlap-add plane (floats); a multiple of 32
  static constexpr int SLOTS = TOUT / 4 + 16;  // y slots per band: slot u + 1 + j for u < TOUT/4
  static constexpr int YP = TOUT / 4 + 20;   // a band's y row: slot at +3, read 20 at a time
  static constexpr int NB = TOUT / 256;      // 256-sample output blocks
};

// The launch's walk over the tiles.  Tiles are numbered item-major; workgroup b takes tiles
// base, base + stride, ... below its end, passing over those with no kept sample.  With a
// workgroup per tile: base = b, stride = the grid, end = all tiles.  When workgroups loop (the
// grid a multiple of 8), the tiles are split into 8 contiguous runs, one per XCD (workgroup b runs
// on XCD b % 8), and the XCD's workgroups take its run in order: neighbouring tiles, which read
// the same boundary frames, then share that XCD's L2.  The stride steps (item, bx) by sq items
// and sr tiles, so no division per step.  Each item's kept samples are [lo, hi) (clamped to its
// samples; item 0 and the last item have their own bounds: the windows of a long request).
struct TailWalk {
  int nbx, batch, ntiles, xcd_run;   // xcd_run: tiles per XCD run, 0 = no split
  int stride, sq, sr;
  int lo_first, lo, hi, hi_last;
};

template <int TOUT>
__global__ void __launch_bounds__(256) tail_kernel(const float *__restrict__ p, long long ldp,
                                                   long long bsp, int L, float *__restrict__ wav,
                                                   long long bsw, const float *__restrict__ cst,
                                                   TailWalk tw) {
  using G = TailGeo<TOUT>;
  constexpr int NG = G::NG, P = G::P, SLOTS = G::SLOTS, YP = G::YP, NB = G::NB;
  static_assert(NB >= 1 && NB <= 4 && TOUT % 256 == 0, "one 256-sample block per wave");
  // s_pl[band][jt][jr]: sample n = 4 jt + (jr & 3) of relative frame (jr >> 2) - jt, so
  // ola[jr] = sum_jt s_pl[band][jt][jr]; s_y[band][slot + 3]
  __shared__ __align__(16) float s_pl[4 * 4 * P];
  __shared__ __align__(16) float s_y[4 * YP];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int lm = lane & 15, lg = lane >> 4;
  const float *hann = cst, *bc = cst + 16, *bs = cst + 160, *hp = cst + 304, *hb = cst + 560;
  const int Ly = 4 * (L - 1);

  // this workgroup's tiles (TailWalk); (item, bx) = divmod(tile, nbx)
  const int b0 = (int) blockIdx.x;
  int tile = tw.xcd_run ? (b0 & 7) * tw.xcd_run + (b0 >> 3) : b0;
  const int tend = tw.xcd_run ? min(((b0 & 7) + 1) * tw.xcd_run, tw.ntiles) : tw.ntiles;
  int item = tile / tw.nbx, bx = tile - item * tw.nbx;
  auto step = [&](int &t, int &it, int &b) {
    t += tw.stride;
    it += tw.sq;
    b += tw.sr;
    if (b >= tw.nbx) {
      b -= tw.nbx;
      it++;
    }
  };
  auto kept_lo = [&](int it) { return it == 0 ? tw.lo_first : tw.lo; };
  auto kept_hi = [&](int it) { return it + 1 == tw.batch ? tw.hi_last : tw.hi; };
  auto to_kept = [&](int &t, int &it, int &b) {
    while (t < tend && !(b * TOUT < kept_hi(it) && b * TOUT + TOUT > kept_lo(it))) step(t, it, b);
  };
  to_kept(tile, item, bx);
  if (tile >= tend) return;

  // reads of one tile: for frame group c of band w, lane (m, g) reads frame t_lo + 16c + m of
  // bins g and g + 4 (magnitude and phase) and, in k group 0, bin 8.  The item's 72 rows are one
  // buffer; a frame outside [0, L) gets an offset past it and reads 0 (the host keeps 72 * ldp
  // floats within 2 GiB); the row steps between the reads are scalar offsets.
  const unsigned nrec = (unsigned) (72 * ldp * 4), ldp4 = (unsigned) (ldp * 4);
  const unsigned ro = (unsigned) (18 * w + lg) * ldp4;
  float ld[NG][6];
  auto issue = [&](int it, int b) {
    const int t_lo = b * (TOUT / 16) - 3;
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        (void *) (p + (long long) it * bsp), (short) 0, (int) nrec, PTK_BUF_WORD3);
#pragma unroll
    for (int c = 0; c < NG; c++) {
      const int tf = t_lo + 16 * c + lm;
      const bool ok = (unsigned) tf < (unsigned) L;
      const unsigned vo = ok ? ro + (unsigned) tf * 4u : PTK_OOB;
      const unsigned vo8 = ok && lg == 0 ? vo + 8u * ldp4 : PTK_OOB;
      ld[c][0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, vo, 0, 0));
      ld[c][1] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, vo, 9 * ldp4, 0));
      ld[c][2] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, vo, 4 * ldp4, 0));
      ld[c][3] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, vo, 13 * ldp4, 0));
      ld[c][4] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, vo8, 0, 0));
      ld[c][5] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, vo8, 9 * ldp4, 0));
    }
  };
  issue(item, bx);

  // B operands, the same for every tile: the irfft basis of this lane's k group with hann[n]
  // folded in, and the synthesis taps (gain 4 folded in: an exact power-of-two scaling) of band
  // lg for output n = 4q + r at each shift s
  float ba[4], bf[19];
  {
    const float h = hann[lm];
    ba[0] = h * bc[lg * 16 + lm];
    ba[1] = h * (lg == 0 ? bc[8 * 16 + lm] : bs[lg * 16 + lm]);
    ba[2] = h * bc[(lg + 4) * 16 + lm];
    ba[3] = h * bs[(lg + 4) * 16 + lm];
    const int q = lm >> 2, r = lm & 3;
#pragma unroll
    for (int s = 0; s < 19; s++) {
      const int j = s - q;
      bf[s] = j >= 0 && j < 16 ? 4.0f * hp[(lg * 4 + r) * 16 + j] : 0.0f;
    }
  }
  const float bias = hb[0];
  // phase B: lane slot = lane + 64 it has jr & 3 = lane & 3, so its window-sum terms hann^2 are
  // fixed.  Every y is ola * (1 / max(wsum, 1e-9)), wsum summed over the valid terms in tap
  // order: the interior value is computed once here, by the same operations.
  const float eps = 1e-9f;
  float hh[4];
#pragma unroll
  for (int jt = 0; jt < 4; jt++) {
    const float h = hann[(lane & 3) + 4 * jt];
    hh[jt] = h * h;
  }
  float ws_in = 0.0f;
#pragma unroll
  for (int jt = 0; jt < 4; jt++) ws_in += hh[jt];
  const float inv_in = 1.0f / (ws_in > eps ? ws_in : eps);
  float *const pl = s_pl + w * 4 * P;        // this wave's band
  float *const yw = s_y + w * YP + 3;

  for (bool first = true;; first = false) {
    const int o0 = bx * TOUT;
    const int t_lo = o0 / 16 - 3;             // frame of relative index 0
    const int i_lo = o0 / 4 - 8;              // y index of slot 0
    // every frame and y slot of the tile inside the sequence: no range tests
    const bool inner = t_lo >= 0 && t_lo + 16 * NG <= L && i_lo >= 0 && i_lo + SLOTS <= Ly;
    // A) band w's frames, 16 per group: spectra into A, 4 MFMAs, the 16 x 16 result into the
    //    overlap-add planes (row 4 lg + i of column lm is sample lm of frame 16c + 4lg + i)
#pragma unroll
    for (int c = 0; c < NG; c++) {
      const int tf = t_lo + 16 * c + lm;
      // the hardware transcendentals: v_exp_f32 is 2^x, v_sin_f32 / v_cos_f32 take revolutions
      // (sin(2 pi x)).  The phase pi * sin(p) in revolutions is sin(p) / 2, within [-1/2, 1/2],
      // so the outer cos / sin need no range reduction.  The inner sin(p) does: p is an
      // unbounded conv output (reduced by rev_of below).
      const float m0 = __builtin_amdgcn_exp2f(ld[c][0] * 1.44269504f);
      const float r0 = 0.5f * __builtin_amdgcn_sinf(rev_of(ld[c][1]));
      const float m1 = __builtin_amdgcn_exp2f(ld[c][2] * 1.44269504f);
      const float r1 = 0.5f * __builtin_amdgcn_sinf(rev_of(ld[c][3]));
      const float m8 = __builtin_amdgcn_exp2f(ld[c][4] * 1.44269504f);
      const float r8 = 0.5f * __builtin_amdgcn_sinf(rev_of(ld[c][5]));
      float a0 = m0 * __builtin_amdgcn_cosf(r0);
      float a1 = lg == 0 ? m8 * __builtin_amdgcn_cosf(r8) : m0 * __builtin_amdgcn_sinf(r0);
      float a2 = m1 * __builtin_amdgcn_cosf(r1);
      float a3 = m1 * __builtin_amdgcn_sinf(r1);
      if (!inner && (unsigned) tf >= (unsigned) L) {   // frames outside the sequence are zero
        a0 = 0.0f;
        a1 = 0.0f;
        a2 = 0.0f;
        a3 = 0.0f;
      }
      f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
      d = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, ba[0], d, 0, 0, 0);
      d = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, ba[1], d, 0, 0, 0);
      d = __builtin_amdgcn_mfma_f32_16x16x4f32(a2, ba[2], d, 0, 0, 0);
      d = __builtin_amdgcn_mfma_f32_16x16x4f32(a3, ba[3], d, 0, 0, 0);
      float *const dst = pl + (lm >> 2) * P + 64 * c + 16 * lg + lm;
#pragma unroll
      for (int i = 0; i < 4; i++) dst[4 * i] = d[i];
    }
    int ntile = tile, nitem = item, nxb = bx;
    step(ntile, nitem, nxb);
    to_kept(ntile, nitem, nxb);
    const bool more = ntile < tend;
    if (more) issue(nitem, nxb);   // in flight through phases B and C
    // the previous tile's phase C read every band's y
    if (!first) __syncthreads();
    // B) band w's y: overlap-add, window-sum normalisation, [8:-8] trim; 0 outside [0, Ly)
    if (inner) {
#pragma unroll
      for (int it = 0; it < (SLOTS + 63) / 64; it++) {
        const int slot = lane + 64 * it, jr = slot + 12;
        if (slot < SLOTS)
          yw[slot] = (((pl[jr] + pl[P + jr]) + pl[2 * P + jr]) + pl[3 * P + jr]) * inv_in;
      }
    } else {
#pragma unroll
      for (int it = 0; it < (SLOTS + 63) / 64; it++) {
        const int slot = lane + 64 * it;
        if (slot < SLOTS) {
          const int jr = slot + 12, i = i_lo + slot;
          float yv = 0.0f;
          if (i >= 0 && i < Ly) {
            const float ola = ((pl[jr] + pl[P + jr]) + pl[2 * P + jr]) + pl[3 * P + jr];
            const int t0 = t_lo + (jr >> 2);    // frame of tap jt is t0 - jt
            float ws = 0.0f;
#pragma unroll
            for (int jt = 0; jt < 4; jt++) ws += (unsigned) (t0 - jt) < (unsigned) L ? hh[jt] : 0.0f;
            yv = ola * (1.0f / (ws > eps ? ws : eps));
          }
          yw[slot] = yv;
        }
      }
    }
    __syncthreads();
    // C) PQMF synthesis of the 256-sample block w: A = y_lg[64w + 4m + 1 + s] (a lane's 20
    //    consecutive values in five 16-byte reads), B = the taps of shift s; the result row
    //    4lg + i, column lm is sample o0 + 256w + 16(4lg + i) + lm
    if (w < NB) {
      const float4 *ya = reinterpret_cast<const float4 *>(s_y + lg * YP + 64 * w + 4 * lm + 4);
      float a[20];
#pragma unroll
      for (int v = 0; v < 5; v++) {
        const float4 x = ya[v];
        a[4 * v] = x.x; a[4 * v + 1] = x.y; a[4 * v + 2] = x.z; a[4 * v + 3] = x.w;
      }
      f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < 19; s++) d = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], bf[s], d, 0, 0, 0);
      // samples outside the item's kept range (which lies inside its samples) get an offset past
      // the buffer: the store is dropped by the range check
      const int lo = kept_lo(item), hi = kept_hi(item);
      const unsigned cnt = hi > lo ? (unsigned) (hi - lo) : 0u;
      const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
          (void *) (wav + (long long) item * bsw), (short) 0, (int) 0x7fffffff, PTK_BUF_WORD3);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int o = o0 + 256 * w + 16 * (4 * lg + i) + lm;
        const unsigned vo = (unsigned) (o - lo) < cnt ? (unsigned) o * 4u : PTK_OOB;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(d[i] + bias), rw, vo, 0, 0);
      }
    }
    if (!more) break;
    tile = ntile;
    item = nitem;
    bx = nxb;
  }
}

template <int TOUT>
static int launch_tail(int batch, const float *p, int64_t ldp, int64_t bsp, int64_t L, float *wav,
                       int64_t bsw, const float *consts, const ptk_emit *em, int grid_knob,
                       hipStream_t s) {
  const int nout = (int) (16 * (L - 1));
  const int nbx = (nout + TOUT - 1) / TOUT;
  const long long ntiles = (long long) nbx * batch;
  if (ntiles > INT_MAX / 2) {
    set_err("ptk_tail: %lld tiles exceed the launch's index range", ntiles);
    return -1;
  }
  // A workgroup per tile while the tiles fit on the chip at once; past that, as many workgroups
  // as are resident, each looping over tiles with the next tile's reads in flight (PTK_TAIL_GRID:
  // -1 = a workgroup per tile, n > 0 = n workgroups).
  static const int resident = [] {
    int ncu = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, 0) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, tail_kernel<TOUT>, 256, 0) !=
            hipSuccess)
      return 0;
    return ncu * per_cu;
  }();
  long long grid = grid_knob > 0 ? grid_knob : (grid_knob < 0 || resident <= 0 ? ntiles : resident);
  if (grid > ntiles) grid = ntiles;
  // looping workgroups split the tiles into one contiguous run per XCD (PTK_TAIL_XCD=0: no split)
  const int xcd_run = grid < ntiles && grid % 8 == 0 && knob(KN_TAIL_XCD)
      ? (int) ((ntiles + 7) / 8) : 0;
  const int stride = xcd_run ? (int) (grid / 8) : (int) grid;
  auto clamp = [nout](int64_t v) { return (int) (v < 0 ? 0 : (v > nout ? nout : v)); };
  const TailWalk tw = {nbx, batch, (int) ntiles, xcd_run, stride, stride / nbx, stride % nbx,
                       clamp(em->lo_first), clamp(em->lo), clamp(em->hi), clamp(em->hi_last)};
  hipLaunchKernelGGL((tail_kernel<TOUT>), dim3((unsigned) grid), dim3(256), 0, s, p,
                     (long long) ldp, (long long) bsp, (int) L, wav, (long long) bsw, consts, tw);
  HCHK(hipGetLastError());
  return 0;
}

extern "C" int ptk_tail_batched(const float *p, int64_t ldp, int64_t bsp, int64_t L, float *wav,
                                int64_t bsw, int batch, const float *consts, const ptk_emit *emit,
                                void *s) {
  if (L < 2) {
    set_err("ptk_tail: need at least 2 frames (got %lld)", (long long) L);
    return -1;
  }
  // 32-bit buffer offsets: an item's 72 rows and its waveform within 2 GiB each
  if (ldp < L || 72 * ldp * 4 > INT32_MAX || 16 * (L - 1) * 4 > INT32_MAX) {
    set_err("ptk_tail: %lld frames (row stride %lld) past the kernel's 32-bit offsets",
            (long long) L, (long long) ldp);
    return -1;
  }
  if (batch <= 0) return 0;
  const long long nout = 16 * (L - 1);
  const ptk_emit all = {0, 0, nout, nout};
  const ptk_emit em = emit ? *emit : all;
  // Tile size: PTK_TAIL_OUT=256 / 512 / 1024 forces one.
  const int oknob = knob(KN_TAIL_OUT), gknob = knob(KN_TAIL_GRID);
  const long long t1k = (nout + 1023) / 1024 * batch, t512 = (nout + 511) / 512 * batch;
  hipStream_t st = (hipStream_t) s;
  const int tout = oknob == 256 || oknob == 512 || oknob == 1024
      ? oknob : (t1k >= 256 ? 1024 : (t512 >= 256 ? 512 : 256));
  if (tout == 1024)
    return launch_tail<1024>(batch, p, ldp, bsp, L, wav, bsw, consts, &em, gknob, st);
  if (tout == 512)
    return launch_tail<512>(batch, p, ldp, bsp, L, wav, bsw, consts, &em, gknob, st);
  return launch_tail<256>(batch, p, ldp, bsp, L, wav, bsw, consts, &em, gknob, st);
}
extern "C" int ptk_tail(const float *p, int64_t ldp, int64_t L, float *wav, const float *consts,
                        void *s) {
  return ptk_tail_batched(p, ldp, 0, L, wav, 0, 1, consts, NULL, s);
}

// ------------------------------------------------------------------------------ MFMA layout probe
__global__ void mfma_probe_kernel(const float *a, const float *b, float *d) {
  const int lane = threadIdx.x;
  f32x16 acc;
  for (int v = 0; v < 16; v++) acc[v] = 0.0f;
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[(lane & 31) * 2 + (lane >> 5)],
                                             b[(lane >> 5) * 32 + (lane & 31)], acc, 0, 0, 0);
  for (int v = 0; v < 16; v++) {
    const int i = 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3), j = lane & 31;
    d[i * 32 + j] = acc[v];
  }
}
extern "C" int ptk_mfma_probe(const float *a, const float *b, float *d, void *s) {
  hipLaunchKernelGGL(mfma_probe_kernel, dim3(1), dim3(64), 0, (hipStream_t) s, a, b, d);
  HCHK(hipGetLastError());
  return 0;
}

// 16x16x4: lane l holds A[l % 16][l / 16] and B[l / 16][l % 16]; value r of its result is
// D[4*(l / 16) + r][l % 16], the layout the tail's products assume
__global__ void mfma16_probe_kernel(const float *a, const float *b, float *d) {
  const int lane = threadIdx.x;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[(lane & 15) * 4 + (lane >> 4)],
                                             b[(lane >> 4) * 16 + (lane & 15)], acc, 0, 0, 0);
  for (int r = 0; r < 4; r++) d[(4 * (lane >> 4) + r) * 16 + (lane & 15)] = acc[r];
}
extern "C" int ptk_mfma16_probe(const float *a, const float *b, float *d, void *s) {
  hipLaunchKernelGGL(mfma16_probe_kernel, dim3(1), dim3(64), 0, (hipStream_t) s, a, b, d);
  HCHK(hipGetLastError());
  return 0;
}
