// Checks of the device memory pool (sisi4s_amd/csrc) on the host: the few HIP
// calls that it makes are replaced here by a device of a set size.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <thread>

#include "../sisi4s_amd/csrc/common.hpp"

namespace {
std::mutex device_m;
std::map<char *, size_t> device;        // allocations (addresses that are never read)
size_t device_size = 0, device_used = 0;
char *next_address = reinterpret_cast<char *>(uintptr_t(1) << 40);
int frees = 0;
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  std::lock_guard<std::mutex> lock(device_m);
  if (device_used + n > device_size) return hipErrorOutOfMemory;
  device_used += n;
  *p = next_address;
  device[next_address] = n;
  next_address += (n + 4095) / 4096 * 4096;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> lock(device_m);
  auto it = device.find(static_cast<char *>(p));
  if (it == device.end()) {
    fprintf(stderr, "hipFree of an address that is not allocated\n");
    abort();
  }
  device_used -= it->second;
  device.erase(it);
  ++frees;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
}

using sisi::Pool;

#define CHECK(c)                                                  \
  do {                                                            \
    if (!(c)) {                                                   \
      fprintf(stderr, "%s:%d: %s\n", __FILE__, __LINE__, #c);     \
      return 1;                                                   \
    }                                                             \
  } while (0)

constexpr size_t MB = size_t(1) << 20;

// What the pool calls cached is what a trim gives back, with small buffers
// (carved out of slabs) in use next to cached ones and with large ones.
static int cached_is_trimmable() {
  device_size = 4096 * MB;
  Pool pool;
  void *a = pool.get(3 * MB), *b = pool.get(3 * MB), *c = pool.get(200 * MB), *d = pool.get(300 * MB);
  pool.put(a);
  pool.put(c);
  size_t before = device_used, cached = pool.cached_bytes();
  pool.trim();
  CHECK(before - device_used == cached);
  CHECK(cached == 200 * MB);  // b holds its slab
  pool.put(b);
  pool.put(d);
  before = device_used;
  cached = pool.cached_bytes();
  pool.trim();
  CHECK(before - device_used == cached && device_used == 0);
  return 0;
}

// The room that a larger buffer left in a slab serves smaller ones later.
static int slab_tails_are_used() {
  device_size = 4096 * MB;
  Pool pool;
  pool.get(40 * MB);  // a slab of 80
  pool.get(41 * MB);  // one of 82
  pool.get(41 * MB);  // its other half
  const size_t used = device_used;
  pool.get(40 * MB);
  CHECK(device_used == used);
  return 0;
}

int main(int argc, char **argv) {
  struct {
    const char *name;
    int (*f)();
  } tests[] = {{"cached_is_trimmable", cached_is_trimmable},
               {"slab_tails_are_used", slab_tails_are_used}};
  for (auto &t : tests)
    if (argc == 2 && std::string(argv[1]) == t.name) return t.f();
  fprintf(stderr, "unknown test\n");
  return 2;
}
