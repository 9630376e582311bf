// device_pool.cpp -- device memory that outlives one call: an index's arrays and the
// workspaces of index builds and column encodings.
//
// hipMalloc and hipFree of such blocks cost as much as the work in them: 0.1 and 0.3 ms a
// block in a fresh process, and about 25 us a megabyte to free once a process has used most
// of the device's memory (a 1e8-row build takes 5.6 GB in 13 blocks and runs 8 ms of
// kernels; encoding a 1e8-row column 2.9 GB in 6 blocks).  Freed blocks are therefore kept
// for the next call of any thread or stream:
//   - a block is given to pool_free only when no queued work can touch it any more, so it
//     can be handed out at once;
//   - at most kPoolBytes are kept on each device, the oldest going back first;
//   - all of a device's kept blocks go back when an allocation of the library fails there
//     (which is then tried again) and when a caller asks for it (rts_device_mem_trim);
//   - a kept block that the device does not take back (hipFree is refused beside some stream
//     captures) stays kept.
// A block's list node is made before the block and moves from list to list with it, so nothing
// here throws into the C entry points that call it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <iterator>
#include <list>
#include <mutex>
#include <new>

#include "device_mem.h"

namespace rts {
namespace {

constexpr size_t kPoolBytes = (size_t)8 << 30;  // kept on each device, at most

// Sizes are rounded up, so that a freed block fits the next call's.
size_t rounded(size_t bytes) {
  const size_t granule = bytes < ((size_t)1 << 20) ? (size_t)64 << 10 : (size_t)2 << 20;
  return (std::max<size_t>(bytes, 1) + granule - 1) / granule * granule;
}

struct Block {
  void *ptr;
  size_t bytes;
  int dev;
};

struct Pool {
  std::mutex mu;
  std::list<Block> kept;  // oldest first
  std::list<Block> in_use;
};

// Never destroyed: blocks may be freed while the process ends, in any order.
Pool &pool() {
  static Pool *p = new Pool;
  return *p;
}

size_t kept_bytes(const Pool &p, int dev) {
  size_t total = 0;
  for (const Block &k : p.kept) total += k.dev == dev ? k.bytes : 0;
  return total;
}

// hipFree of kept blocks taken off the list, outside the lock (hipFree waits for the device).
void give_back(std::list<Block> &blocks) {
  for (auto b = blocks.begin(); b != blocks.end();) {
    auto next = std::next(b);
    if (hipFree(b->ptr) == hipSuccess) blocks.erase(b);
    b = next;
  }
  if (blocks.empty()) return;
  (void)hipGetLastError();
  Pool &p = pool();
  std::lock_guard<std::mutex> lock(p.mu);
  p.kept.splice(p.kept.begin(), blocks);
}

}  // namespace

void pool_trim(int dev) {
  std::list<Block> out;
  {
    Pool &p = pool();
    std::lock_guard<std::mutex> lock(p.mu);
    for (auto it = p.kept.begin(); it != p.kept.end();) {
      auto next = std::next(it);
      if (it->dev == dev) out.splice(out.end(), p.kept, it);
      it = next;
    }
  }
  give_back(out);
}

size_t pool_kept(int dev) {
  Pool &p = pool();
  std::lock_guard<std::mutex> lock(p.mu);
  return kept_bytes(p, dev);
}

bool device_wait() {
  void *p = nullptr;
  if (hipMalloc(&p, 1) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return hipFree(p) == hipSuccess;  // 0.7 us both on an idle device
}

hipError_t device_malloc(void **ptr, size_t bytes) {
  hipError_t e = hipMalloc(ptr, bytes);
  int dev = 0;
  if (e != hipErrorOutOfMemory || hipGetDevice(&dev) != hipSuccess) return e;
  (void)hipGetLastError();  // the first try's error is not the caller's
  pool_trim(dev);
  return hipMalloc(ptr, bytes);
}

hipError_t pool_alloc(void **ptr, size_t bytes) {
  *ptr = nullptr;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  bytes = rounded(bytes);
  Pool &p = pool();
  {
    std::lock_guard<std::mutex> lock(p.mu);
    auto best = p.kept.end();  // the smallest block that holds it and wastes at most a quarter
    for (auto it = p.kept.begin(); it != p.kept.end(); ++it)
      if (it->dev == dev && it->bytes >= bytes && it->bytes <= bytes + bytes / 4 &&
          (best == p.kept.end() || it->bytes < best->bytes))
        best = it;
    if (best != p.kept.end()) {
      *ptr = best->ptr;
      p.in_use.splice(p.in_use.end(), p.kept, best);
      return hipSuccess;
    }
  }
  std::list<Block> block;
  try {
    block.push_back(Block{nullptr, bytes, dev});
  } catch (const std::bad_alloc &) {
    return hipErrorOutOfMemory;
  }
  e = device_malloc(&block.front().ptr, bytes);
  if (e != hipSuccess) return e;
  *ptr = block.front().ptr;
  std::lock_guard<std::mutex> lock(p.mu);
  p.in_use.splice(p.in_use.end(), block);
  return hipSuccess;
}

void pool_free(void *ptr, bool idle) {
  if (!ptr) return;
  std::list<Block> out;
  {
    Pool &p = pool();
    std::lock_guard<std::mutex> lock(p.mu);
    auto it = std::find_if(p.in_use.begin(), p.in_use.end(), [&](const Block &b) { return b.ptr == ptr; });
    if (it == p.in_use.end()) return;
    if (!idle) {
      out.splice(out.end(), p.in_use, it);
    } else {
      const int dev = it->dev;
      p.kept.splice(p.kept.end(), p.in_use, it);
      size_t total = kept_bytes(p, dev);
      for (auto k = p.kept.begin(); k != p.kept.end() && total > kPoolBytes;) {
        auto next = std::next(k);
        if (k->dev == dev) {
          total -= k->bytes;
          out.splice(out.end(), p.kept, k);
        }
        k = next;
      }
    }
  }
  if (idle)
    give_back(out);
  else
    (void)hipFree(out.front().ptr);  // the device may still use it: hipFree waits
}

}  // namespace rts
