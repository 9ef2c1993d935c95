// Stream-ordered workspaces of single calls.
//
// The device's default pool gives its memory back to the system whenever the
// GPU is waited for, so a program that waits after each call paid for mapping
// the workspace again each time. The library has a pool of its own per device,
// which keeps up to kKeepBytes of freed memory (under a hundredth of the
// device's) until jc_release_workspaces or the end of the process; larger
// workspaces are mapped in part, 0.4 of 16.2 ms for the 5.7 GB of RMAT-22. Blocks
// go from one stream to another in the runtime's order, as in the default pool.
// While a stream is captured the allocation is a node of the graph, as before.
// Calls that are waited for, us: weighted RMAT of 200003 vertices (0.26 GB) 1115
// -> 735, Chung-Lu 2^20 3080 -> 2869, 16M draws ingested 2322 -> 1937.
#include <hip/hip_runtime.h>

#include <mutex>

#include "../../include/jaccard_amd.h"
#include "jc_internal.hpp"

namespace jc {
namespace {

constexpr uint64_t kKeepBytes = 2ull << 30;
constexpr int kMaxDevices = 64;
std::mutex g_mu;
hipMemPool_t g_pool[kMaxDevices] = {};
bool g_none[kMaxDevices] = {};  // no pool could be made: the default one serves

// The pool of a device, or nullptr.
hipMemPool_t pool_of(int dev) {
  if (dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_mu);
  if (!g_pool[dev] && !g_none[dev]) {
    hipMemPoolProps props{};
    props.allocType = hipMemAllocationTypePinned;
    props.handleTypes = hipMemHandleTypeNone;
    props.location.type = hipMemLocationTypeDevice;
    props.location.id = dev;
    hipMemPool_t p = nullptr;
    uint64_t keep = kKeepBytes;
    if (hipMemPoolCreate(&p, &props) == hipSuccess &&
        hipMemPoolSetAttribute(p, hipMemPoolAttrReleaseThreshold, &keep) == hipSuccess) {
      g_pool[dev] = p;
    } else {
      (void)hipGetLastError();
      if (p) (void)hipMemPoolDestroy(p);
      g_none[dev] = true;
    }
  }
  return g_pool[dev];
}

}  // namespace

hipError_t call_alloc(void** p, size_t bytes, hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  int dev = 0;
  if (hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone ||
      (s ? hipStreamGetDevice(s, &dev) : hipGetDevice(&dev)) != hipSuccess) {
    (void)hipGetLastError();
    return hipMallocAsync(p, bytes, s);
  }
  hipMemPool_t pool = pool_of(dev);
  if (!pool) return hipMallocAsync(p, bytes, s);
  hipError_t e = hipMallocFromPoolAsync(p, bytes, pool, s);
  if (e == hipSuccess) return e;
  (void)hipGetLastError();
  (void)hipMemPoolTrimTo(pool, 0);  // what is kept may be in blocks too small
  return hipMallocAsync(p, bytes, s);
}

}  // namespace jc

extern "C" int jc_release_workspaces(void) {
  std::lock_guard<std::mutex> lock(jc::g_mu);
  for (hipMemPool_t p : jc::g_pool) {
    if (!p) continue;
    const hipError_t e = hipMemPoolTrimTo(p, 0);
    if (e != hipSuccess) return jc::note_hip_error(e);
  }
  return JC_OK;
}
