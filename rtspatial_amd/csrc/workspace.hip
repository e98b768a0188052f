// Device scratch of query, sort and serve calls, kept between calls.
//
// A call leases a block for work on its stream and gives it back when the
// work is queued; the block goes to the next call whose work may follow it:
// one on the same stream, or on any stream once the block's event has passed.
// The stream-ordered pool that stood here reuses a freed block only for a
// request of nearly its size and maps memory again otherwise, which cost more
// than the calls: 1M within queries took 116 ms (5.4 ms of kernels), 20k
// intersects queries 8.7 ms (1.9 ms).
//
// Kept blocks are bounded: 1/16 of the device's memory while an index lives on
// it, kIdleBytes otherwise, least recently used given back first (which, like
// any free, waits for the device). The last index's end, rts_release_scratch
// and an allocation of the library's that finds the device full
// (device_alloc: the index's own arrays too) give back all of them. A stream
// that is being captured gets graph-owned memory instead (stream-ordered from
// the device's default pool), since a replay may run at any time.
#include <algorithm>
#include <list>
#include <mutex>

#include "rts_internal.h"

namespace rts {
namespace {

constexpr int kMaxDevices = 64;
constexpr size_t kIdleBytes = 256ull << 20;

struct Kept {
  void* p;
  size_t bytes;
  hipEvent_t done;
  hipStream_t stream;  // of the last lease
};

struct Device {
  std::mutex mu;
  std::list<Kept> kept;  // least recently used first
  size_t bytes = 0;      // of `kept`
  size_t limit = 0;      // with an index alive
  int indexes = 0;
};

Device& device(int dev) {
  static Device* all = new Device[kMaxDevices];  // never destroyed: leases may outlive static teardown
  return all[dev];
}

// Sizes are rounded to an eighth of their power of two (at most 64 MiB), so
// that calls of nearly equal sizes share blocks.
size_t rounded(size_t bytes) {
  size_t step = 64 << 10;
  while (step * 16 <= bytes && step < (64ull << 20)) step <<= 1;
  return (bytes + step - 1) / step * step;
}

void give_back(const Kept& k) {
  (void)hipEventSynchronize(k.done);
  (void)hipEventDestroy(k.done);
  (void)hipFree(k.p);
}

// Gives back kept blocks, oldest first, until at most `most` bytes are kept.
void trim(Device& d, size_t most) {
  while (d.bytes > most && !d.kept.empty()) {
    const Kept k = d.kept.front();
    d.kept.pop_front();
    d.bytes -= k.bytes;
    give_back(k);
  }
}

void give_back_all(Device& d) {
  Relaxed relaxed;
  std::lock_guard<std::mutex> lk(d.mu);
  trim(d, 0);
}

}  // namespace

hipError_t workspace_lease(size_t bytes, hipStream_t stream, Lease* out) {
  *out = Lease{};
  if (bytes == 0) return hipSuccess;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  out->device = dev;
  out->stream = stream;
  if (capturing(stream)) {
    e = hipMallocAsync(&out->p, bytes, stream);
    if (e == hipSuccess) out->stream_ordered = true;
    return e;
  }
  const size_t need = rounded(bytes);
  Relaxed relaxed;
  Device& d = device(dev);
  std::unique_lock<std::mutex> lk(d.mu);
  // The smallest block that fits, is not twice as large, and is free for
  // this stream.
  auto best = d.kept.end();
  for (auto it = d.kept.begin(); it != d.kept.end(); ++it) {
    if (it->bytes < need || it->bytes / 2 > need) continue;
    if (best != d.kept.end() && it->bytes >= best->bytes) continue;
    if (it->stream != stream && hipEventQuery(it->done) != hipSuccess) continue;
    best = it;
  }
  (void)hipGetLastError();  // hipErrorNotReady is no error of the caller's
  if (best != d.kept.end()) {
    // The same handle may name a new stream: order it after the event (work
    // on one stream is in order already).
    if (best->stream == stream && stream != nullptr && hipEventQuery(best->done) != hipSuccess) {
      (void)hipGetLastError();
      e = hipStreamWaitEvent(stream, best->done, 0);
      if (e != hipSuccess) return e;
    }
    out->p = best->p;
    out->bytes = best->bytes;
    out->done = best->done;
    d.bytes -= best->bytes;
    d.kept.erase(best);
    return hipSuccess;
  }
  lk.unlock();
  e = device_alloc(&out->p, need);
  if (e != hipSuccess) {
    out->p = nullptr;
    return e;
  }
  out->bytes = need;
  e = hipEventCreateWithFlags(&out->done, hipEventDisableTiming);
  if (e != hipSuccess) {
    (void)hipFree(out->p);
    *out = Lease{};
  }
  return e;
}

hipError_t device_alloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  int dev = 0;
  if (e == hipErrorOutOfMemory && hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices) {
    (void)hipGetLastError();
    give_back_all(device(dev));
    e = hipMalloc(p, bytes);
  }
  // The caller reports e; it is not to turn up at the program's next HIP call.
  if (e != hipSuccess) (void)hipGetLastError();
  return e;
}

void workspace_return(Lease* lease) {
  const Lease l = *lease;
  *lease = Lease{};
  if (!l.p) return;
  if (l.stream_ordered) {
    (void)hipFreeAsync(l.p, l.stream);
    return;
  }
  Relaxed relaxed;
  Device& d = device(l.device);
  // An event that cannot be recorded leaves the order unknown: wait instead.
  if (hipEventRecord(l.done, l.stream) != hipSuccess) {
    (void)hipGetLastError();
    (void)hipDeviceSynchronize();
  }
  std::lock_guard<std::mutex> lk(d.mu);
  if (!d.limit) {
    size_t free_bytes = 0, total = 0;
    if (hipMemGetInfo(&free_bytes, &total) == hipSuccess) d.limit = total / 16;
    d.limit = std::max(d.limit, kIdleBytes);
  }
  d.kept.push_back(Kept{l.p, l.bytes, l.done, l.stream});
  d.bytes += l.bytes;
  trim(d, d.indexes ? d.limit : kIdleBytes);
}

void workspace_index_begin(int dev) {
  if (dev < 0 || dev >= kMaxDevices) return;
  std::lock_guard<std::mutex> lk(device(dev).mu);
  device(dev).indexes++;
}

void workspace_index_end(int dev) {
  if (dev < 0 || dev >= kMaxDevices) return;
  Relaxed relaxed;
  Device& d = device(dev);
  std::lock_guard<std::mutex> lk(d.mu);
  if (--d.indexes == 0) trim(d, 0);
}

}  // namespace rts

extern "C" int rts_release_scratch(void) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= rts::kMaxDevices) {
    rts::set_error("rts_release_scratch: no HIP device");
    return RTS_ERR_MISSING;
  }
  rts::give_back_all(rts::device(dev));
  return RTS_OK;
}
