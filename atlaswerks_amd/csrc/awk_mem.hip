// awk_mem.hip -- device memory that outlives a handle or a call.
//
// dev_alloc / dev_free: the buffers of operators and of greedy and LDMM iterators (an
// atlas's own slabs, the network's and the trainer's are plain allocations).  A handle's
// allocation and release map and unmap its pages (160 x 192 x 144 greedy iterator: 1.1
// ms to create, 1.0 to destroy, against 0.19 ms per iteration), and a multiscale run
// makes one per level.  Released blocks are kept for the next handle that wants the
// same sizes: at most 1 GiB per device in blocks of up to 512 MiB, the oldest given back
// first.  A block is put away only once the work on it is done: the null stream is waited
// for where its handle used no other, else the device (as hipFree waits).  So whoever
// takes it next, on any thread or stream, finds no work on it.
//
// scratch_alloc / scratch_free: stream-ordered scratch of one call, from a pool that
// keeps up to 512 MiB between calls; the runtime's default pool gives everything back
// at each synchronisation and the next call pays for the mapping (a 256^3 splat that
// is waited for: 650 us with it, 260 from the pool).
//
// What is kept is given back, and the allocation tried once more, when any of this
// library's allocations (device_malloc among them) finds the device full.  Other
// allocators in the process cannot ask for it: awk_release_memory does.
#include <mutex>
#include <new>
#include <unordered_map>
#include <vector>

#include "awk_common.h"

namespace awk {

namespace {
constexpr size_t kCacheMax = 1ull << 30, kCacheBlockMax = 512ull << 20, kScratchKeep = 512ull << 20;
constexpr int kMaxDev = 64;

struct Block {
  void *p;
  size_t size;
  int dev;
};
struct Cache {
  std::mutex mu;
  std::vector<Block> idle;  // oldest first
  std::unordered_map<void *, Block> live;
  size_t held[kMaxDev] = {};
  hipMemPool_t pool[kMaxDev] = {};
  bool pool_tried[kMaxDev] = {};
};
Cache &cache() {  // never destroyed: handles may be released at the process's end
  static Cache *c = new Cache();
  return *c;
}
// Waits for the device as hipFree does, which a relaxed capture allows:
// hipDeviceSynchronize invalidates it.  0.7 us on a device long idle, about 30 just after
// a handle's last work, so blocks that only the null stream used wait for that stream
// (three-level warp 160 x 192 x 144 3.17 -> 3.07 ms).
bool device_idle() {
  void *p = nullptr;
  if (hipMalloc(&p, 64) == hipSuccess && hipFree(p) == hipSuccess) return true;
  (void)hipGetLastError();
  return false;
}
// Everything kept on device dev goes back to the runtime (the lock is held).
void release_kept(Cache &c, int dev) {
  // scratch that is free in stream order only is free then (hipFree below waits as well)
  if (!device_idle() && c.idle.empty()) (void)hipDeviceSynchronize();
  for (size_t i = 0; i < c.idle.size();)
    if (c.idle[i].dev == dev) {
      (void)hipFree(c.idle[i].p);
      c.held[dev] -= c.idle[i].size;
      c.idle.erase(c.idle.begin() + i);
    } else {
      ++i;
    }
  if (c.pool[dev]) (void)hipMemPoolTrimTo(c.pool[dev], 0);
}
// alloc() once more with nothing kept if the device was full.
template <class F>
hipError_t or_release(F alloc, int dev) {
  hipError_t e = alloc();
  if (e != hipErrorOutOfMemory || dev < 0 || dev >= kMaxDev) return e;
  Cache &c = cache();
  std::lock_guard<std::mutex> lock(c.mu);
  (void)hipGetLastError();
  release_kept(c, dev);
  return alloc();
}
// A block handed out, with room to put it away later: dev_free allocates nothing, so it
// throws nothing.  False when host memory has run out.
bool hold(Cache &c, const Block &b) {
  try {
    if (c.idle.capacity() < c.idle.size() + c.live.size() + 1) c.idle.reserve(2 * (c.idle.size() + c.live.size() + 1));
    c.live[b.p] = b;
    return true;
  } catch (const std::bad_alloc &) {
    return false;
  }
}
size_t block_size(size_t bytes) {
  const size_t unit = bytes < (1u << 20) ? 4096 : 65536;
  return (bytes + unit - 1) / unit * unit;
}
}  // namespace

hipError_t device_malloc_bytes(void **p, size_t bytes) {
  *p = nullptr;
  int dev = -1;
  if (hipError_t e = hipGetDevice(&dev)) return e;
  return or_release([&] { return hipMalloc(p, bytes); }, dev);
}

hipError_t dev_alloc_bytes(void **p, size_t bytes) {
  if (!bytes) return device_malloc_bytes(p, bytes);
  *p = nullptr;
  int dev = -1;
  if (hipError_t e = hipGetDevice(&dev)) return e;
  const size_t want = block_size(bytes);
  Cache &c = cache();
  {
    // the same size only: a larger block would hold more than the handle needs
    std::lock_guard<std::mutex> lock(c.mu);
    for (size_t i = 0; i < c.idle.size(); ++i) {
      const Block b = c.idle[i];
      if (b.dev != dev || b.size != want) continue;
      if (!hold(c, b)) return hipErrorOutOfMemory;
      c.idle.erase(c.idle.begin() + i);
      c.held[dev] -= b.size;
      *p = b.p;
      return hipSuccess;
    }
  }
  if (hipError_t e = or_release([&] { return hipMalloc(p, want); }, dev)) return e;
  std::lock_guard<std::mutex> lock(c.mu);
  if (hold(c, Block{*p, want, dev})) return hipSuccess;
  (void)hipFree(*p);
  *p = nullptr;
  return hipErrorOutOfMemory;
}

void dev_free(void *const *blocks, int n, bool null_only) {
  bool any = false;
  for (int i = 0; i < n; ++i) any = any || blocks[i];
  if (!any) return;
  int dev = -1;
  const bool idle = hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDev &&
                    (null_only ? hipStreamSynchronize(nullptr) == hipSuccess : device_idle());
  Cache &c = cache();
  std::lock_guard<std::mutex> lock(c.mu);
  for (int i = 0; i < n; ++i) {
    if (!blocks[i]) continue;
    auto it = c.live.find(blocks[i]);
    const bool known = it != c.live.end();
    const Block b = known ? it->second : Block{blocks[i], 0, -1};
    if (known) c.live.erase(it);
    if (!known || !idle || b.dev != dev || b.size > kCacheBlockMax) {
      (void)hipFree(b.p);
      continue;
    }
    c.idle.push_back(b);
    c.held[dev] += b.size;
    for (size_t k = 0; c.held[dev] > kCacheMax && k < c.idle.size();)
      if (c.idle[k].dev == dev) {
        (void)hipFree(c.idle[k].p);
        c.held[dev] -= c.idle[k].size;
        c.idle.erase(c.idle.begin() + k);
      } else {
        ++k;
      }
  }
}

hipError_t scratch_alloc_bytes(void **p, size_t bytes, hipStream_t s) {
  *p = nullptr;
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  const bool capturing = hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone;
  if (capturing) (void)hipGetLastError();
  hipMemPool_t pool = nullptr;
  if (!capturing && dev >= 0 && dev < kMaxDev) {
    Cache &c = cache();
    std::lock_guard<std::mutex> lock(c.mu);
    if (!c.pool_tried[dev]) {
      c.pool_tried[dev] = true;
      hipMemPoolProps props = {};
      props.allocType = hipMemAllocationTypePinned;
      props.location.type = hipMemLocationTypeDevice;
      props.location.id = dev;
      unsigned long long keep = kScratchKeep;
      if (hipMemPoolCreate(&c.pool[dev], &props) != hipSuccess ||
          hipMemPoolSetAttribute(c.pool[dev], hipMemPoolAttrReleaseThreshold, &keep) != hipSuccess) {
        c.pool[dev] = nullptr;
        (void)hipGetLastError();
      }
    }
    pool = c.pool[dev];
  }
  if (capturing) return hipMallocAsync(p, bytes, s);
  if (!pool) return or_release([&] { return hipMallocAsync(p, bytes, s); }, dev);
  return or_release([&] { return hipMallocFromPoolAsync(p, bytes, pool, s); }, dev);
}

hipError_t scratch_free(void *p, hipStream_t s) { return hipFreeAsync(p, s); }

}  // namespace awk

using namespace awk;

extern "C" awk_status awk_release_memory(void) {
  int dev = -1;
  AWK_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDev) return AWK_OK;  // (none is kept there)
  Cache &c = cache();
  std::lock_guard<std::mutex> lock(c.mu);
  release_kept(c, dev);
  return AWK_OK;
}
