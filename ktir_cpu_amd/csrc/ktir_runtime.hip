// Runtime half of the C ABI: device selection, the library stream, memory,
// events and error reporting.  The simulated HBM of the reference
// (memory.py:311-398) is a single device arena allocated through these calls by
// the host runtime; the reference's sparse dict of NumPy arrays becomes plain
// device memory.
//
// Small copies between host and device (arguments, launch tables, results of
// a call on a few KB) go through a pinned ring and a copy kernel on the library
// stream: an upload is queued without waiting for it, a list of results is read
// back behind one wait, and errors found on the device are a word of pinned
// memory that needs no copy.  Each hipMemcpyAsync from or to pageable memory and
// its wait took 15 to 23 us; a call on 24 KB (vector_add of 4096) makes three uploads
// and three downloads and read the error word twice: 442 -> 246 us for the call.
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include "ktir_common.h"

namespace ktir {

static thread_local char g_err[1024] = "";
static hipStream_t g_stream = nullptr;
static int* g_err_flag = nullptr;
static int g_device = -1;

// The pinned ring.  A part is handed out again only after the stream has
// drained, under the mutex that also covers what is queued from it.
constexpr uint64_t RING = 1 << 20, SMALL_COPY = 64 << 10, SMALL_LIST = 256 << 10;
// One copy that is waited for is faster through the runtime from here on (16 KB
// up 18.7 us and down 22.1 there, 14.9 and 14.2 through the ring; 24 KB 10.4 and
// 10.5 against 15.2 and 14.6); queued without a wait the ring takes 6.4 us.
constexpr uint64_t ONE_COPY = 16 << 10;
// Coherent, whatever the runtime's default: the host writes a part again that an
// earlier kernel has read, and the next kernel must not find the old bytes in
// the device's cache; the same goes for the error word.
constexpr unsigned PINNED = hipHostMallocPortable | hipHostMallocCoherent;
static std::mutex g_ring_mutex;
static uint8_t* g_ring = nullptr;
static uint64_t g_ring_head = 0;

constexpr int COPY_PARTS = 8;
typedef uint32_t copy4 __attribute__((ext_vector_type(4)));
struct CopyParts {
  uint64_t dst[COPY_PARTS], src[COPY_PARTS];
  uint32_t bytes[COPY_PARTS];
};

// part blockIdx.y: 16 bytes per thread where both ends allow it
__global__ __launch_bounds__(256) void copy_parts(const CopyParts p) {
  const uint64_t dst = p.dst[blockIdx.y], src = p.src[blockIdx.y];
  const uint32_t n = p.bytes[blockIdx.y], at = (blockIdx.x * 256 + threadIdx.x) * 16;
  if (at >= n) return;
  if (!((dst | src) & 15) && at + 16 <= n) {
    *(KTIR_G(copy4)*)(dst + at) = *(const KTIR_G(copy4)*)(src + at);
    return;
  }
  const uint32_t end = at + 16 < n ? at + 16 : n;
  for (uint32_t i = at; i < end; ++i) ((KTIR_G(uint8_t)*)dst)[i] = ((const KTIR_G(uint8_t)*)src)[i];
}

int set_error(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

hipStream_t stream() { return g_stream; }
int* device_error_flag() { return g_err_flag; }

}  // namespace ktir

using namespace ktir;

extern "C" const char* ktir_last_error(void) { return g_err; }

extern "C" int ktir_init(int device) {
  if (g_device == device && g_stream) return KTIR_OK;
  int n = 0;
  KTIR_HIP_CHECK(hipGetDeviceCount(&n));
  if (device < 0 || device >= n) return set_error(KTIR_E_ARG, "ktir_init: device %d of %d", device, n);
  KTIR_HIP_CHECK(hipSetDevice(device));
  KTIR_HIP_CHECK(hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking));
  if (!g_err_flag) {
    KTIR_HIP_CHECK(hipHostMalloc((void**)&g_err_flag, sizeof(int), PINNED));
    *g_err_flag = 0;
  }
  g_device = device;
  return rmw_scratch_setup(device);
}

extern "C" int ktir_shutdown(void) {
  if (!g_stream) return KTIR_OK;
  KTIR_HIP_CHECK(hipStreamSynchronize(g_stream));
  KTIR_HIP_CHECK(hipHostFree(g_err_flag));
  g_err_flag = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_ring_mutex);
    if (g_ring) KTIR_HIP_CHECK(hipHostFree(g_ring));
    g_ring = nullptr;
    g_ring_head = 0;
  }
  KTIR_HIP_CHECK(hipStreamDestroy(g_stream));
  g_stream = nullptr;
  g_device = -1;
  return KTIR_OK;
}

extern "C" int ktir_device_info(int* cu_count, int* clock_khz, int64_t* hbm_bytes, char* name, int name_len) {
  hipDeviceProp_t p;
  int dev = g_device < 0 ? 0 : g_device;
  KTIR_HIP_CHECK(hipGetDeviceProperties(&p, dev));
  if (cu_count) *cu_count = p.multiProcessorCount;
  if (clock_khz) *clock_khz = p.clockRate;
  if (hbm_bytes) *hbm_bytes = (int64_t)p.totalGlobalMem;
  if (name && name_len > 0) {
    snprintf(name, name_len, "%s (%s)", p.name, p.gcnArchName);
  }
  return KTIR_OK;
}

extern "C" int ktir_malloc(uint64_t bytes, uint64_t* dptr) {
  void* p = nullptr;
  KTIR_HIP_CHECK(hipMalloc(&p, bytes ? bytes : 1));
  *dptr = (uint64_t)p;
  return KTIR_OK;
}

extern "C" int ktir_free(uint64_t dptr) {
  KTIR_HIP_CHECK(hipStreamSynchronize(g_stream));
  KTIR_HIP_CHECK(hipFree((void*)dptr));
  return KTIR_OK;
}

// `bytes` of the ring, 256-byte aligned (the mutex held); null: no ring
static uint8_t* ring_take(uint64_t bytes) {
  if (!g_ring) {
    if (hipHostMalloc((void**)&g_ring, RING, PINNED) != hipSuccess) {
      (void)hipGetLastError();
      g_ring = nullptr;
      return nullptr;
    }
    g_ring_head = 0;
  }
  bytes = (bytes + 255) & ~255ull;
  if (g_ring_head + bytes > RING) {
    if (hipStreamSynchronize(g_stream) != hipSuccess) return nullptr;
    g_ring_head = 0;
  }
  uint8_t* p = g_ring + g_ring_head;
  g_ring_head += bytes;
  return p;
}

// whether copies of these sizes go through the ring (never while the stream is
// being captured: a replay would read what the ring then holds)
static bool ring_fits(int n, const uint64_t* bytes) {
  uint64_t sum = 0;
  for (int i = 0; i < n; ++i) {
    if (bytes[i] > SMALL_COPY) return false;
    sum += (bytes[i] + 255) & ~255ull;
  }
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return sum && sum <= SMALL_LIST && hipStreamIsCapturing(g_stream, &st) == hipSuccess && st == hipStreamCaptureStatusNone;
}

// queue the parts' copies between device addresses and `ring` (parts one after another, 256-byte aligned)
static int ring_copy(int n, const uint64_t* dev, uint8_t* ring, const uint64_t* bytes, bool to_device) {
  for (int i = 0; i < n;) {
    CopyParts p;
    int k = 0;
    uint32_t most = 0;
    for (; i < n && k < COPY_PARTS; ++i) {
      if (bytes[i]) {
        p.dst[k] = to_device ? dev[i] : (uint64_t)ring;
        p.src[k] = to_device ? (uint64_t)ring : dev[i];
        p.bytes[k] = (uint32_t)bytes[i];
        if (p.bytes[k] > most) most = p.bytes[k];
        ++k;
      }
      ring += (bytes[i] + 255) & ~255ull;
    }
    if (k) hipLaunchKernelGGL(copy_parts, dim3((most + 4095) / 4096, k), dim3(256), 0, g_stream, p);
  }
  KTIR_HIP_CHECK(hipGetLastError());
  return KTIR_OK;
}

extern "C" int ktir_upload_list(int n, const uint64_t* dst, const void* const* src, const uint64_t* bytes) {
  if (n < 0 || (n && (!dst || !src || !bytes))) return set_error(KTIR_E_ARG, "ktir_upload_list: bad list");
  if (ring_fits(n, bytes)) {
    std::lock_guard<std::mutex> lock(g_ring_mutex);
    uint64_t sum = 0;
    for (int i = 0; i < n; ++i) sum += (bytes[i] + 255) & ~255ull;
    if (uint8_t* ring = ring_take(sum)) {
      uint8_t* p = ring;
      for (int i = 0; i < n; ++i) {
        if (bytes[i]) memcpy(p, src[i], bytes[i]);
        p += (bytes[i] + 255) & ~255ull;
      }
      return ring_copy(n, dst, ring, bytes, true);
    }
  }
  bool any = false;
  for (int i = 0; i < n; ++i) {
    if (!bytes[i]) continue;
    KTIR_HIP_CHECK(hipMemcpyAsync((void*)dst[i], src[i], bytes[i], hipMemcpyHostToDevice, g_stream));
    any = true;
  }
  if (any) KTIR_HIP_CHECK(hipStreamSynchronize(g_stream));
  return KTIR_OK;
}

extern "C" int ktir_download_list(int n, void* const* dst, const uint64_t* src, const uint64_t* bytes) {
  if (n < 0 || (n && (!dst || !src || !bytes))) return set_error(KTIR_E_ARG, "ktir_download_list: bad list");
  if (!(n == 1 && bytes[0] > ONE_COPY) && ring_fits(n, bytes)) {
    std::lock_guard<std::mutex> lock(g_ring_mutex);
    uint64_t sum = 0;
    for (int i = 0; i < n; ++i) sum += (bytes[i] + 255) & ~255ull;
    if (uint8_t* ring = ring_take(sum)) {
      const int rc = ring_copy(n, src, ring, bytes, false);
      if (rc != KTIR_OK) return rc;
      KTIR_HIP_CHECK(hipStreamSynchronize(g_stream));
      for (int i = 0; i < n; ++i) {
        if (bytes[i]) memcpy(dst[i], ring, bytes[i]);
        ring += (bytes[i] + 255) & ~255ull;
      }
      return KTIR_OK;
    }
  }
  bool any = false;
  for (int i = 0; i < n; ++i) {
    if (!bytes[i]) continue;
    KTIR_HIP_CHECK(hipMemcpyAsync(dst[i], (const void*)src[i], bytes[i], hipMemcpyDeviceToHost, g_stream));
    any = true;
  }
  if (any) KTIR_HIP_CHECK(hipStreamSynchronize(g_stream));
  return KTIR_OK;
}

extern "C" int ktir_memcpy_h2d(uint64_t dst, const void* src, uint64_t bytes) {
  if (!bytes) return KTIR_OK;
  if (bytes > ONE_COPY) {
    KTIR_HIP_CHECK(hipMemcpyAsync((void*)dst, src, bytes, hipMemcpyHostToDevice, g_stream));
  } else {
    const int rc = ktir_upload_list(1, &dst, &src, &bytes);
    if (rc != KTIR_OK) return rc;
  }
  KTIR_HIP_CHECK(hipStreamSynchronize(g_stream));   // in place for other streams too
  return KTIR_OK;
}

extern "C" int ktir_memcpy_d2h(void* dst, uint64_t src, uint64_t bytes) {
  return ktir_download_list(1, &dst, &src, &bytes);
}

extern "C" int ktir_memcpy_d2d(uint64_t dst, uint64_t src, uint64_t bytes) {
  if (!bytes) return KTIR_OK;
  KTIR_HIP_CHECK(hipMemcpyAsync((void*)dst, (const void*)src, bytes, hipMemcpyDeviceToDevice, g_stream));
  return KTIR_OK;
}

extern "C" int ktir_memset(uint64_t dst, int value, uint64_t bytes) {
  if (!bytes) return KTIR_OK;
  KTIR_HIP_CHECK(hipMemsetAsync((void*)dst, value, bytes, g_stream));
  return KTIR_OK;
}

extern "C" int ktir_sync(void) {
  KTIR_HIP_CHECK(hipStreamSynchronize(g_stream));
  return KTIR_OK;
}

extern "C" int ktir_check_error_flag(void) {
  KTIR_HIP_CHECK(hipStreamSynchronize(g_stream));
  volatile int* flag = g_err_flag;
  if (flag && *flag) {
    *flag = 0;
    return set_error(KTIR_E_INDEX, "indirect index is negative");
  }
  return KTIR_OK;
}

// Timing events: no system-scope fence when one is recorded, so recording
// it does not write back and invalidate the caches between the launches it
// separates (elapsed times only need the timestamps; ktir_sync or
// ktir_event_elapsed_ms waits for completion).
extern "C" int ktir_event_create(uint64_t* ev) {
  hipEvent_t e;
  KTIR_HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableSystemFence));
  *ev = (uint64_t)e;
  return KTIR_OK;
}

extern "C" int ktir_event_record(uint64_t ev) {
  KTIR_HIP_CHECK(hipEventRecord((hipEvent_t)ev, g_stream));
  return KTIR_OK;
}

extern "C" int ktir_event_elapsed_ms(uint64_t start, uint64_t stop, float* ms) {
  KTIR_HIP_CHECK(hipEventSynchronize((hipEvent_t)stop));
  KTIR_HIP_CHECK(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop));
  return KTIR_OK;
}

extern "C" int ktir_event_destroy(uint64_t ev) {
  KTIR_HIP_CHECK(hipEventDestroy((hipEvent_t)ev));
  return KTIR_OK;
}
