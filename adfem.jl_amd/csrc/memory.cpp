// Device memory of the library's buffers (DevBuf): hipMalloc with a bounded
// cache of released blocks in front of it.
//
// A mesh, its system and a solver's workspace are some ninety allocations, a
// new sparse pattern fifty with as many releases; hipMalloc and hipFree of
// blocks of a few MB cost 50 - 300 us each on MI355X, more than the kernels
// between them (Mesh + bcnode + DirichletSystem at 300^2: 15.1 -> 6.6 ms).
//
// A released block waits for the device before it is cached, as hipFree
// does, so whoever gets it next -- any stream, any thread -- cannot meet work
// still queued on it.  Blocks above CACHE_BLOCK, or past CACHE_TOTAL in all,
// go back to the driver at once; everything cached does when an allocation
// fails, and by admfem_release_memory.
#include <map>
#include <mutex>
#include <vector>

#include "internal.h"

namespace admfem {

namespace {

constexpr size_t CACHE_BLOCK = (size_t)64 << 20, CACHE_TOTAL = (size_t)512 << 20;

// a request's size class: powers of two up to 64 KiB, then eighths of them;
// blocks that are never cached have their own size
size_t size_class(size_t bytes) {
  if (bytes > CACHE_BLOCK) return bytes;
  size_t p = 256;
  while (p < bytes) p <<= 1;
  if (p <= (size_t)64 << 10) return p;
  const size_t step = p >> 4;  // the power below p, in eighths
  return (bytes + step - 1) / step * step;
}

struct Cache {
  std::mutex mu;
  std::multimap<std::pair<int, size_t>, void *> blocks;  // (device, class)
  size_t total = 0;
};
Cache &cache() {
  static Cache *c = new Cache();  // lives until the process ends
  return *c;
}

}  // namespace

void release_device_memory() {
  Cache &c = cache();
  std::multimap<std::pair<int, size_t>, void *> out;
  {
    std::lock_guard<std::mutex> g(c.mu);
    out.swap(c.blocks);
    c.total = 0;
  }
  for (auto &b : out) (void)hipFree(b.second);
}

size_t device_available() {
  size_t avail = 0, total = 0;
  int dev = -1;
  HIPCHECK(hipMemGetInfo(&avail, &total));
  HIPCHECK(hipGetDevice(&dev));
  Cache &c = cache();
  std::lock_guard<std::mutex> g(c.mu);
  for (auto &b : c.blocks)
    if (b.first.first == dev) avail += b.first.second;
  return avail;
}

void *device_alloc(size_t bytes, int &device) {
  HIPCHECK(hipGetDevice(&device));
  const size_t cls = size_class(bytes);
  Cache &c = cache();
  {
    std::lock_guard<std::mutex> g(c.mu);
    auto it = c.blocks.find({device, cls});
    if (it != c.blocks.end()) {
      void *p = it->second;
      c.blocks.erase(it);
      c.total -= cls;
      return p;
    }
  }
  void *p = nullptr;
  if (hipMalloc(&p, cls) != hipSuccess) {
    (void)hipGetLastError();
    release_device_memory();
    if (hipMalloc(&p, cls) != hipSuccess) {
      (void)hipGetLastError();
      throw OutOfMemory{{ADMFEM_ERR_HIP, "out of device memory: " + std::to_string(cls) +
                                             " bytes"}};
    }
  }
  return p;
}

void device_free(void *p, size_t bytes, int device) {
  const size_t cls = size_class(bytes);
  int dev = -1;
  // (a device other than the current one, a block too large, or a wait that
  // is refused -- a thread capturing a graph: back to the driver)
  if (cls <= CACHE_BLOCK && hipGetDevice(&dev) == hipSuccess && dev == device &&
      hipDeviceSynchronize() == hipSuccess) {
    Cache &c = cache();
    std::lock_guard<std::mutex> g(c.mu);
    if (c.total + cls <= CACHE_TOTAL) {
      c.blocks.emplace(std::make_pair(device, cls), p);
      c.total += cls;
      return;
    }
  }
  (void)hipGetLastError();
  (void)hipFree(p);
}

// ------------------------------------------------------------- host slots

namespace {
struct Slots {
  std::mutex mu;
  std::vector<void *> free_;  // at most as many as calls ever ran at once
};
Slots &slots() {
  static Slots *s = new Slots();  // lives until the process ends
  return *s;
}
}  // namespace

HostSlot::HostSlot(hipStream_t stream) : p(nullptr), st(stream) {
  {
    Slots &s = slots();
    std::lock_guard<std::mutex> g(s.mu);
    if (!s.free_.empty()) {
      p = s.free_.back();
      s.free_.pop_back();
      return;
    }
  }
  HIPCHECK(hipHostMalloc(&p, 64, hipHostMallocPortable));
}

HostSlot::~HostSlot() {
  if (pending) (void)hipStreamSynchronize(st);  // (an error between read and wait)
  Slots &s = slots();
  std::lock_guard<std::mutex> g(s.mu);
  s.free_.push_back(p);
}

}  // namespace admfem
