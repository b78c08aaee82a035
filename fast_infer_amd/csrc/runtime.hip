// Library-wide host helpers: error strings, version, the CU count per device, the XCD-group
// check and arrival counters of the kernels that share partial results within an XCD, and the
// MFMA layout self-test.
#include <stdarg.h>

#include <atomic>
#include <mutex>

#include "common.h"

namespace fi {

static thread_local char g_error[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

void clear_error() { g_error[0] = '\0'; }

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: kernel launch failed: %s", what, hipGetErrorString(e));
    return FI_ERR_HIP;
  }
  return FI_OK;
}

// Compute units of the device that runs `stream` (the current device for the null stream),
// queried once per device and cached.
int device_cu_count(hipStream_t stream) {
  constexpr int kMaxDevices = 64;
  static std::atomic<int> cache[kMaxDevices];
  int dev = -1;
  if (stream != nullptr) {
    hipDevice_t d;
    if (hipStreamGetDevice(stream, &d) == hipSuccess) dev = (int)d;
  }
  if (dev < 0 && hipGetDevice(&dev) != hipSuccess) dev = -1;
  if (dev >= 0 && dev < kMaxDevices) {
    const int v = cache[dev].load(std::memory_order_relaxed);
    if (v > 0) return v;
  }
  int cus = 0;
  if (dev < 0 || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus <= 0)
    return 256;  // MI355X
  if (dev < kMaxDevices) cache[dev].store(cus, std::memory_order_relaxed);
  return cus;
}

// ---------------------------------------------------------------------------------------
// XCD groups.  The dispatcher deals consecutive workgroups of a launch to the XCDs in turn, so
// workgroups whose block ids are congruent modulo 8 run on one XCD and share its L2: kernels
// that pass partial sums between such workgroups (through stores, an L2 atomic counter and
// L1-bypassing loads) use this only after one probe launch per device has shown it to hold.

constexpr int kMaxDevices = 64;
constexpr int kProbeBlocks = 2048;
__device__ unsigned g_xcd_probe[kProbeBlocks];

__global__ __launch_bounds__(64) void xcd_probe_kernel(unsigned* out) {
  if (threadIdx.x == 0) {
    unsigned x;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(x));
    out[blockIdx.x] = x & 0xf;
  }
}

// Arrival counters, zero at load and left zero by every launch.  Launches on one stream follow
// one another, so they share the stream's set (one per stream, in order of first use, up to
// kXcdStreams streams).  A graph may be replayed beside any stream and any other graph: each
// capture gets sets of its own, one for every stream taking part (what is captured on one
// stream forms a chain in the graph; a program that rewires a capture's dependencies by hand has
// to keep that order), from a part of the array that is only ever handed out once: 16 MiB, 2 to 8
// KiB a set; captures past it use the second launch.  A set for each launch lasted 146 captures
// of a 28-layer step with two such calls a layer; this lasts 8192.
constexpr int kXcdStreams = 16;
constexpr int kXcdSet = 8 * kXcdCounters;
constexpr int kXcdCaptured = 4 << 20;
__device__ __attribute__((aligned(256))) unsigned g_xcd_counters[kXcdStreams * kXcdSet + kXcdCaptured];

struct XcdCapture {  // the set of one stream in one capture
  hipStream_t st = nullptr;
  unsigned long long id = 0;
  unsigned* counters = nullptr;
  int stride = 0;
};

struct XcdDevice {
  int state = 0;  // 0: not probed, 1: groups share an XCD, -1: they do not (or no answer)
  unsigned* counters = nullptr;
  hipStream_t streams[kXcdStreams] = {};
  int used = 0;      // streams with a set
  int captured = 0;  // counters handed to captures
  XcdCapture captures[kXcdStreams];  // the latest, a place per stream (any one may be taken over)
  int next = 0;
};

static std::mutex& xcd_mutex() {
  static std::mutex mu;
  return mu;
}

static XcdDevice& xcd_device(int dev) {
  static XcdDevice devs[kMaxDevices];
  return devs[dev];
}

static int stream_device(hipStream_t st) {
  hipDevice_t d;
  if (hipStreamGetDevice(st, &d) != hipSuccess) return -1;
  return (int)d < kMaxDevices ? (int)d : -1;
}

// One probe launch on `st`: every block records its XCC_ID into g_xcd_probe (no allocation),
// read back with a synchronous copy.  Called with the device of `st` current.
static bool xcd_probe(hipStream_t st) {
  void* d = nullptr;
  if (hipGetSymbolAddress(&d, HIP_SYMBOL(g_xcd_probe)) != hipSuccess || !d) return false;
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  (void)hipThreadExchangeStreamCaptureMode(&mode);
  static unsigned h[kProbeBlocks];
  hipLaunchKernelGGL(xcd_probe_kernel, dim3(kProbeBlocks), dim3(64), 0, st, (unsigned*)d);
  bool ok = hipGetLastError() == hipSuccess &&
            hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, st) == hipSuccess &&
            hipStreamSynchronize(st) == hipSuccess;
  for (int i = 8; ok && i < kProbeBlocks; ++i) ok = h[i] == h[i & 7];
  (void)hipThreadExchangeStreamCaptureMode(&mode);
  return ok;
}

// Whether workgroups whose block ids are congruent modulo 8 run on one XCD of `dev` (one probe
// launch and a synchronous copy on `st` at the device's first call; false, and not yet probed,
// while `st` is being captured).
static bool xcd_ready(XcdDevice& xd, int dev, hipStream_t st) {
  if (xd.state == 0) {
    // the probe synchronizes: not while `st` is being captured or an error is pending
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipPeekAtLastError() != hipSuccess) return false;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    if (cs != hipStreamCaptureStatusNone) return false;
    int cur = -1;
    if (hipGetDevice(&cur) != hipSuccess) return false;
    if (cur != dev && hipSetDevice(dev) != hipSuccess) return false;
    void* addr = nullptr;
    const bool ok = hipGetSymbolAddress(&addr, HIP_SYMBOL(g_xcd_counters)) == hipSuccess && addr;
    xd.counters = (unsigned*)addr;
    xd.state = ok && xcd_probe(st) ? 1 : -1;
    if (cur != dev) (void)hipSetDevice(cur);
  }
  return xd.state == 1;
}

unsigned* xcd_counters(hipStream_t st, int per_group, int* stride) {
  // hipStreamPerThread names another stream in every thread
  if (per_group > kXcdCounters || st == hipStreamPerThread) return nullptr;
  const int dev = stream_device(st);
  if (dev < 0) return nullptr;
  std::lock_guard<std::mutex> lock(xcd_mutex());
  XcdDevice& xd = xcd_device(dev);
  if (!xcd_ready(xd, dev, st)) return nullptr;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (st != nullptr && hipStreamGetCaptureInfo(st, &cs, &id) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  if (cs == hipStreamCaptureStatusInvalidated) return nullptr;
  if (cs == hipStreamCaptureStatusActive) {
    int i = 0;
    while (i < kXcdStreams && xd.captures[i].st != st) ++i;
    if (i == kXcdStreams) {
      i = xd.next;
      xd.next = (i + 1) % kXcdStreams;
    }
    XcdCapture& c = xd.captures[i];
    if (c.st != st || c.id != id || c.stride < per_group) {
      const int need = (per_group + 63) / 64 * 64;
      if (xd.captured + 8 * need > kXcdCaptured) return nullptr;
      c = XcdCapture{st, id, xd.counters + kXcdStreams * kXcdSet + xd.captured, need};
      xd.captured += 8 * need;
    }
    *stride = c.stride;
    return c.counters;
  }
  *stride = kXcdCounters;
  int i = 0;
  while (i < xd.used && xd.streams[i] != st) ++i;
  if (i == xd.used) {
    if (i == kXcdStreams) return nullptr;
    xd.streams[xd.used++] = st;
  }
  return xd.counters + i * kXcdSet;
}

// One wave: c = mfma16x16x32(a, b, 0) with the lane-major fragments of the header.
__global__ __launch_bounds__(64) void selftest_mfma_kernel(const half8* a, const half8* b,
                                                           floatx4* c) {
  const int lane = threadIdx.x;
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  acc = mfma16x16x32(a[lane], b[lane], acc);
  c[lane] = acc;
}

}  // namespace fi

extern "C" int fi_version(void) { return 100; }

extern "C" const char* fi_last_error(void) { return fi::g_error; }

extern "C" int fi_selftest_mfma_f16(const void* a, const void* b, void* c, void* stream) {
  fi::clear_error();
  if (!a || !b || !c) {
    fi::set_error("fi_selftest_mfma_f16: null pointer");
    return FI_ERR_INVALID;
  }
  hipLaunchKernelGGL(fi::selftest_mfma_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream,
                     (const fi::half8*)a, (const fi::half8*)b, (fi::floatx4*)c);
  return fi::check_launch("fi_selftest_mfma_f16");
}
