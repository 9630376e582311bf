// pool_test.cpp -- the pool of device memory (device_pool.cpp) over a device that this file plays:
// what is kept, given back and refused, and no host memory.
#include <stdio.h>
#include <stdlib.h>

#include <hip/hip_runtime.h>

#include <map>
#include <new>

#include "device_mem.h"

static std::map<void *, size_t> device;  // blocks that the device has given
static size_t device_bytes = 0, device_limit = (size_t)1 << 40;
static bool refuse_free = false, no_host_memory = false;
static char *next_address = (char *)0x100000000000;

void *operator new(size_t n) {
  if (no_host_memory) throw std::bad_alloc();
  if (void *p = malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

extern "C" hipError_t hipMalloc(void **p, size_t n) {
  if (device_bytes + n > device_limit) return hipErrorOutOfMemory;
  const bool host = no_host_memory;
  no_host_memory = false;
  *p = next_address;
  next_address += n + 4096;
  device[*p] = n;
  no_host_memory = host;
  device_bytes += n;
  return hipSuccess;
}
extern "C" hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  if (refuse_free) return hipErrorStreamCaptureUnsupported;
  auto it = device.find(p);
  if (it == device.end()) {
    printf("freed twice, or never given\n");
    exit(1);
  }
  device_bytes -= it->second;
  device.erase(it);
  return hipSuccess;
}
extern "C" hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { return hipSuccess; }

#define CHECK(x)                                    \
  do {                                              \
    if (!(x)) {                                     \
      printf("line %d: %s\n", __LINE__, #x);        \
      return 1;                                     \
    }                                               \
  } while (0)

int main() {
  using namespace rts;
  const size_t mb = (size_t)1 << 20, gb = mb << 10;
  void *a = nullptr, *b = nullptr, *c = nullptr;
  // a freed block serves a call of like size, not one that wastes more than a quarter of it
  CHECK(pool_alloc(&a, 100 * mb) == hipSuccess);
  pool_free(a, true);
  CHECK(pool_kept(0) == 100 * mb && pool_kept(1) == 0);
  CHECK(pool_alloc(&b, 90 * mb) == hipSuccess && b == a && pool_kept(0) == 0);
  pool_free(b, true);
  CHECK(pool_alloc(&b, 70 * mb) == hipSuccess && b != a);
  // one that work may still use goes back to the device at once
  pool_free(b, false);
  CHECK(device.count(b) == 0 && pool_kept(0) == 100 * mb);
  // the device's memory runs out: what is kept goes back, and the call gets it
  device_limit = 150 * mb;
  CHECK(pool_alloc(&b, 140 * mb) == hipSuccess && pool_kept(0) == 0 && device.count(a) == 0);
  CHECK(pool_alloc(&c, 20 * mb) == hipErrorOutOfMemory && c == nullptr);
  CHECK(device_malloc(&c, 20 * mb) == hipErrorOutOfMemory);
  pool_free(b, true);
  CHECK(device_malloc(&c, 20 * mb) == hipSuccess && pool_kept(0) == 0);
  CHECK(hipFree(c) == hipSuccess);
  device_limit = (size_t)1 << 40;
  // at most 8 GB are kept, the oldest go first
  void *blocks[6];
  for (void *&p : blocks) CHECK(pool_alloc(&p, 3 * gb) == hipSuccess);
  for (void *p : blocks) pool_free(p, true);
  CHECK(pool_kept(0) == 6 * gb && device.count(blocks[3]) == 0 && device.count(blocks[4]) && device.count(blocks[5]));
  // a device that takes nothing back for a while: the blocks are still the pool's
  refuse_free = true;
  pool_trim(0);
  CHECK(pool_kept(0) == 6 * gb);
  CHECK(pool_alloc(&a, 3 * gb) == hipSuccess && pool_alloc(&b, 3 * gb) == hipSuccess && pool_alloc(&c, 3 * gb) == hipSuccess);
  pool_free(a, true), pool_free(b, true), pool_free(c, true);
  CHECK(pool_kept(0) == 9 * gb);
  CHECK(!device_wait());
  refuse_free = false;
  CHECK(device_wait());
  CHECK(pool_alloc(&a, mb) == hipSuccess);
  pool_free(a, true);
  CHECK(pool_kept(0) <= 8 * gb);
  pool_trim(0);
  CHECK(pool_kept(0) == 0);
  // no host memory: kept blocks are still given and taken, others refused, and nothing is lost
  CHECK(pool_alloc(&a, 10 * mb) == hipSuccess && pool_alloc(&b, 50 * mb) == hipSuccess);
  pool_free(a, true);
  no_host_memory = true;
  CHECK(pool_alloc(&a, 10 * mb) == hipSuccess);
  CHECK(pool_alloc(&c, 10 * mb) == hipErrorOutOfMemory);
  pool_free(a, true);
  pool_free(b, false);
  pool_trim(0);
  no_host_memory = false;
  CHECK(device.size() == 1 && device_bytes == 1);  // device_wait's, whose hipFree was refused
  printf("pool ok\n");
  return 0;
}
