// Workspaces of single calls.
//
// A call's workspace has to be memory that is mapped already. Fresh memory costs
// little only until a process has been through the device's memory once; then
// the system clears what it hands out, at some 25 GB/s, and a call that is waited
// for and so gives its workspace back every time waits for that as well. Measured
// on RMAT-22 (5.65 GB): 100 to 200 ms a call, with single ones of 2 s, for 16 of
// work; a stream of calls on graphs of 2^14 to 2^20 vertices, 1450 -> 50 to 300 a
// second. A pool of the runtime does not help there: its blocks serve requests of
// their own size only.
//
// So the library keeps a few blocks per device, each for one call at a time and
// for any size up to its own. A block is the caller's from get() to release(),
// which records an event on the call's stream; the next call's stream waits for
// that event. Calls on one stream share a block that grows to their largest;
// a call that meets only blocks whose work is still under way on other streams
// takes one more, so streams overlap as before. All blocks of a device together
// hold kKeepBytes at most (the 5.65 GB of RMAT-22 and room for a second stream's),
// until jc_release_workspaces or the end of the process. Beyond that and while a
// stream is captured the allocation is the runtime's, stream-ordered.
//
// All of it comes from the device's default pool. Memory that a thread took from
// a pool of the library's own while another thread captured a call (with its
// allocation as a node of the graph) left that graph without effect from its second replay
// on; with the default pool every replay is right.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "../../include/jaccard_amd.h"
#include "jc_internal.hpp"

namespace jc {
namespace {

constexpr size_t kKeepBytes = size_t(8) << 30;
// A workspace that a call can do without is not taken fresh above this: the
// clearing (2.6 ms) then outweighs what the oriented engine saves on graphs that
// small, and more so above.
constexpr size_t kFreshBytes = size_t(64) << 20;
// A call that a program makes once per graph leaves no more than this behind.
constexpr size_t kOnceBytes = size_t(2) << 30;
constexpr size_t kGrain = size_t(2) << 20;
constexpr int kBlocks = 4;
constexpr int kMaxDevices = 64;

struct Block {
  void* p = nullptr;
  size_t bytes = 0;
  hipEvent_t done = nullptr;      // recorded behind the last call's work
  hipStream_t last = nullptr;     // that call's stream (never used but to compare)
  bool taken = false;
  bool pending = false;           // done was recorded and not seen to be over
};

struct Device {
  std::mutex mu;
  hipStream_t stream = nullptr;   // jc_release_workspaces frees on it
  Block block[kBlocks];
};
Device g_dev[kMaxDevices];

// Another thread may be capturing in the global mode, which forbids these calls
// although none of them touches its stream.
struct Relaxed {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// Whether no call has the block and its last work is over.
bool idle(Block& b) {
  if (b.taken) return false;
  if (b.pending) {
    if (hipEventQuery(b.done) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    b.pending = false;
  }
  return true;
}

// Gives an idle block's memory back, behind what is on s.
void drop(Block& b, hipStream_t s) {
  if (b.p) (void)hipFreeAsync(b.p, s);
  b.p = nullptr;
  b.bytes = 0;
}

// A block of at least `bytes` for work on s, or nullptr. grow: also one that has
// to be mapped anew.
Block* take(Device& d, size_t bytes, hipStream_t s, bool grow) {
  std::lock_guard<std::mutex> lock(d.mu);
  // usable now: this stream's own, whose work comes before what is added, and idle ones
  Block* own = nullptr;
  Block* fit = nullptr;
  Block* any = nullptr;
  size_t held = 0;
  for (Block& b : d.block) {
    held += b.bytes;
    if (b.taken) continue;
    if (b.p && b.last == s) {
      if (!own || b.bytes > own->bytes) own = &b;
    } else if (idle(b)) {
      if (b.bytes >= bytes && (!fit || b.bytes < fit->bytes)) fit = &b;
      if (!any || b.bytes > any->bytes) any = &b;
    }
  }
  Block* b = own && own->bytes >= bytes ? own : fit ? fit : own ? own : any;
  if (!b || (b->bytes < bytes && !grow)) return nullptr;
  // the work it was last used for, also where the handle of s was another
  // stream's before (asked first: a wait for what is over still costs the stream
  // a few us)
  if (!idle(*b) && hipStreamWaitEvent(s, b->done, 0) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  if (b->bytes < bytes) {
    if (!b->done && hipEventCreateWithFlags(&b->done, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      b->done = nullptr;
      return nullptr;
    }
    size_t rest = held - b->bytes;
    for (Block& o : d.block) {
      if (&o == b || !o.p || rest + bytes <= kKeepBytes) continue;
      if (o.last == s && !o.taken && o.pending && hipStreamWaitEvent(s, o.done, 0) == hipSuccess) o.pending = false;
      if (!idle(o)) continue;
      rest -= o.bytes;
      drop(o, s);
    }
    if (rest + bytes > kKeepBytes) return nullptr;
    // a little more than asked for, so that a slow growth is a few steps
    size_t want = std::max(bytes, b->bytes + b->bytes / 4);
    want = std::min((want + kGrain - 1) / kGrain * kGrain, std::max(bytes, (kKeepBytes - rest) / kGrain * kGrain));
    drop(*b, s);
    b->pending = false;
    if (hipMallocAsync(&b->p, want, s) != hipSuccess) {
      (void)hipGetLastError();
      b->p = nullptr;
      return nullptr;
    }
    b->bytes = want;
  }
  b->taken = true;
  return b;
}

// Gives back to the system what no call of the device is using.
hipError_t release_idle(Device& d, int dev) {
  std::lock_guard<std::mutex> lock(d.mu);
  if (std::none_of(d.block, d.block + kBlocks, [](const Block& b) { return b.p != nullptr; })) return hipSuccess;
  int before = 0;
  hipError_t e = hipGetDevice(&before);
  if (e != hipSuccess) return e;
  if ((e = hipSetDevice(dev)) != hipSuccess) return e;
  if (!d.stream) e = hipStreamCreateWithFlags(&d.stream, hipStreamNonBlocking);
  if (e == hipSuccess) {
    for (Block& b : d.block)
      if (b.p && idle(b)) drop(b, d.stream);
    // (the default pool gives back what is free when a stream is waited for)
    e = hipStreamSynchronize(d.stream);
  }
  (void)hipSetDevice(before);
  return e;
}

}  // namespace

hipError_t CallBuf::get(size_t bytes, hipStream_t stream, Use use) {
  release();
  s = stream;
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  int dev = 0;
  if (hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone ||
      (s ? hipStreamGetDevice(s, &dev) : hipGetDevice(&dev)) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    (void)hipGetLastError();
    return hipMallocAsync(&p, bytes, s);
  }
  Relaxed relaxed;
  Device& d = g_dev[dev];
  if (bytes <= kKeepBytes) {
    if (Block* b = take(d, bytes, s, use != kOnce || bytes <= kOnceBytes)) {
      block = b;
      device = dev;
      p = b->p;
      return hipSuccess;
    }
  }
  if (use == kOptional && bytes > kFreshBytes) return hipErrorOutOfMemory;
  hipError_t e = hipMallocAsync(&p, bytes, s);
  if (e == hipSuccess) return e;
  (void)hipGetLastError();
  p = nullptr;
  if (release_idle(d, dev) != hipSuccess) (void)hipGetLastError();
  e = hipMallocAsync(&p, bytes, s);
  if (e != hipSuccess) p = nullptr;
  return e;
}

void CallBuf::release() {
  if (!p) return;
  if (block) {
    Relaxed relaxed;
    Block& b = *static_cast<Block*>(block);
    std::lock_guard<std::mutex> lock(g_dev[device].mu);
    b.last = s;
    b.pending = hipEventRecord(b.done, s) == hipSuccess;
    if (!b.pending) {
      (void)hipGetLastError();
      (void)hipStreamSynchronize(s);
    }
    b.taken = false;
    block = nullptr;
  } else {
    (void)hipFreeAsync(p, s);
  }
  p = nullptr;
}

}  // namespace jc

extern "C" int jc_release_workspaces(void) {
  jc::Relaxed relaxed;
  for (int i = 0; i < jc::kMaxDevices; ++i) {
    const hipError_t e = jc::release_idle(jc::g_dev[i], i);
    if (e != hipSuccess) return jc::note_hip_error(e);
  }
  return JC_OK;
}
