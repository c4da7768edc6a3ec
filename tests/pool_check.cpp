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
hipError_t hipMemGetInfo(size_t *free_b, size_t *total_b) {
  std::lock_guard<std::mutex> lock(device_m);
  *free_b = device_size - device_used;
  *total_b = device_size;
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

static bool fails(Pool &pool, size_t bytes) {
  try {
    pool.get(bytes);
  } catch (const sisi::Error &e) {
    return e.code == SISI_ERR_ALLOC;
  }
  return false;
}

// The block is kept for the next use; a larger one replaces it.
static int block_is_kept() {
  device_size = 1000 * MB;
  Pool pool;
  void *a = pool.take_block(600 * MB);
  CHECK(a && !pool.take_block(100 * MB));
  pool.return_block();
  CHECK(pool.cached_bytes() == 600 * MB);
  CHECK(pool.take_block(500 * MB) == a && frees == 0);
  pool.return_block();
  CHECK(pool.take_block(700 * MB) && device_used == 700 * MB);
  return 0;
}

// A block that fits a slab comes out of one and goes back to the free lists.
static int small_blocks_are_buffers() {
  device_size = 1000 * MB;
  Pool pool;
  pool.get(2 * MB);
  const size_t used = device_used;
  void *a = pool.take_block(4 * MB);
  CHECK(a && device_used == used && !pool.block_lost() && !pool.block_carved());
  pool.return_block();
  CHECK(pool.get(4 * MB) == a && pool.idle_block() == 0);
  return 0;
}

// An allocation of the same pool takes the lent block, but not one in use.
static int block_yields_to_its_pool() {
  device_size = 1000 * MB;
  Pool pool;
  CHECK(pool.take_block(600 * MB));
  pool.begin_use();
  CHECK(fails(pool, 500 * MB) && !pool.block_lost());
  pool.end_use();
  CHECK(pool.get(500 * MB) && pool.block_lost());
  pool.return_block();
  CHECK(!pool.block_lost() && device_used == 500 * MB);
  CHECK(!pool.take_block(600 * MB) && pool.take_block(400 * MB));
  return 0;
}

// Buffers come from the device while a quarter of it stays free, then out of
// the idle block, and when that has no room from the device again.
static int quarter_stays_free() {
  device_size = 1000 * MB;
  Pool pool;
  void *a = pool.take_block(300 * MB);
  pool.get(100 * MB);
  pool.return_block();
  CHECK(pool.get(350 * MB) && device_used == 750 * MB);
  CHECK(pool.get(200 * MB) == a && device_used == 750 * MB);
  CHECK(pool.get(200 * MB) && device_used == 950 * MB);
  return 0;
}

// On a full device buffers come out of the idle block, which is whole again
// (and only then can be had) with the last of them back.
static int block_is_carved() {
  device_size = 1000 * MB;
  Pool pool;
  void *a = pool.take_block(600 * MB);
  void *b = pool.get(400 * MB);
  pool.return_block();
  void *c = pool.get(300 * MB), *d = pool.get(100 * MB);
  CHECK(b && c == a && frees == 0 && device_used == 1000 * MB);
  CHECK(!pool.take_block(600 * MB));
  pool.put(c);
  CHECK(pool.get(300 * MB) == c && !pool.take_block(600 * MB));
  pool.put(c);
  pool.put(d);
  CHECK(pool.take_block(600 * MB) == a);
  CHECK(fails(pool, 700 * MB));  // takes the block, too small all the same
  CHECK(pool.block_lost());
  return 0;
}

// What comes back to the block joins: a buffer larger than each of them, and
// all of it counts as cached.
static int block_ranges_join() {
  device_size = 1000 * MB;
  Pool pool;
  char *a = static_cast<char *>(pool.take_block(600 * MB));
  pool.get(400 * MB);
  pool.return_block();
  void *b[4];
  for (int k = 0; k < 4; ++k) b[k] = pool.get(150 * MB);
  CHECK(b[3] == a + 450 * MB && pool.cached_bytes() == 0);
  pool.put(b[2]);
  pool.put(b[0]);
  pool.put(b[1]);
  CHECK(pool.cached_bytes() == 450 * MB);
  void *c = pool.get(440 * MB), *d = pool.get(10 * MB);
  CHECK(c == a && d && fails(pool, 100 * MB));
  pool.put(c);
  pool.put(b[3]);
  CHECK(pool.block_carved() && pool.idle_block() == 0);
  pool.put(d);
  CHECK(pool.get(590 * MB) == a);
  return 0;
}

// Buffers that a captured graph uses hold the block.
static int block_and_captures() {
  device_size = 1000 * MB;
  Pool pool;
  pool.take_block(600 * MB);
  pool.get(400 * MB);
  pool.return_block();
  pool.begin_capture();
  void *c = pool.get(300 * MB);
  pool.put(c);
  std::vector<void *> held = pool.end_capture();
  CHECK(held.size() == 1 && held[0] == c && !pool.take_block(600 * MB));
  void *d = pool.get(300 * MB);
  CHECK(d != c);
  pool.put(d);
  pool.release(held);
  CHECK(pool.take_block(600 * MB) == c);
  return 0;
}

// A buffer carved before a capture and given back in it: whole at its end.
static int block_given_back_in_a_capture() {
  device_size = 1000 * MB;
  Pool pool;
  void *a = pool.take_block(600 * MB);
  pool.get(400 * MB);
  pool.return_block();
  void *c = pool.get(300 * MB);
  pool.begin_capture();
  pool.put(c);
  pool.release(pool.end_capture());
  CHECK(pool.take_block(600 * MB) == a);
  return 0;
}

// A trim in the course of a capture leaves what captured launches use: a
// buffer of its own, one in a slab, one in the block.
static int trim_in_a_capture() {
  device_size = 1000 * MB;
  Pool pool;
  pool.begin_capture();
  void *a = pool.get(100 * MB), *b = pool.get(1 * MB);
  pool.put(a);
  pool.put(b);
  CHECK(fails(pool, 950 * MB));
  std::vector<void *> held = pool.end_capture();
  CHECK(held.size() == 2 && device_used == 108 * MB);
  CHECK(fails(pool, 950 * MB));
  pool.release(held);
  CHECK(pool.get(950 * MB));
  pool.release_all();
  void *c = pool.take_block(600 * MB);
  pool.get(400 * MB);
  pool.return_block();
  pool.begin_capture();
  CHECK(pool.get(300 * MB) == c);
  pool.put(c);
  CHECK(fails(pool, 550 * MB));
  held = pool.end_capture();
  CHECK(held.size() == 1 && device_used == 1000 * MB);
  pool.release(held);
  CHECK(pool.get(550 * MB));
  return 0;
}

// Another pool's allocation takes the block, lent or idle, and waits for the
// end of its use.
static int block_yields_to_other_pools() {
  device_size = 1000 * MB;
  Pool a, b;
  CHECK(a.take_block(600 * MB));
  a.return_block();
  void *p = b.get(500 * MB);
  CHECK(p && !a.block_lost() && device_used == 500 * MB);
  b.put(p);
  b.trim();
  CHECK(a.take_block(600 * MB));
  p = b.get(500 * MB);
  CHECK(p && a.block_lost());
  b.put(p);
  b.trim();
  a.return_block();
  CHECK(a.take_block(600 * MB));
  a.begin_use();
  CHECK(fails(b, 500 * MB));
  std::thread t([&] {
    std::this_thread::sleep_for(std::chrono::milliseconds(100));
    a.end_use();
  });
  p = b.get(500 * MB);
  t.join();
  CHECK(p && a.block_lost());
  return 0;
}

// Threads that use, give up and take blocks on a device that holds less than
// all of them want.
static int block_from_threads() {
  device_size = 1500 * MB;
  std::atomic<int> used{0}, lost{0}, refused{0};
  auto run = [&](int seed) {
    Pool pool;
    unsigned r = unsigned(seed);
    std::vector<void *> mine;
    bool lent = false;
    for (int k = 0; k < 3000; ++k) {
      r = r * 1664525u + 1013904223u;
      pool.begin_use();
      if (lent && pool.block_lost()) {
        pool.return_block();
        lent = false;
        ++lost;
      }
      if (!lent) lent = pool.take_block(400 * MB) != nullptr;
      if (lent) ++used;
      pool.end_use();
      try {
        if (mine.size() < 3) mine.push_back(pool.get((100 + (r >> 24)) * MB));
      } catch (const sisi::Error &) {
        ++refused;
      }
      if (mine.size() == 3 || (r & 64)) {
        for (void *p : mine) pool.put(p);
        mine.clear();
        if (r & 128) pool.trim();
      }
      if (lent && (r & 256)) {
        pool.return_block();
        lent = false;
      }
    }
  };
  std::vector<std::thread> t;
  for (int k = 0; k < 3; ++k) t.emplace_back(run, k + 1);
  for (auto &x : t) x.join();
  printf("used %d lost %d refused %d\n", used.load(), lost.load(), refused.load());
  CHECK(used > 0 && device_used == 0);
  return 0;
}

int main(int argc, char **argv) {
  struct {
    const char *name;
    int (*f)();
  } tests[] = {{"cached_is_trimmable", cached_is_trimmable},
               {"slab_tails_are_used", slab_tails_are_used},
               {"block_is_kept", block_is_kept},
               {"small_blocks_are_buffers", small_blocks_are_buffers},
               {"block_yields_to_its_pool", block_yields_to_its_pool},
               {"quarter_stays_free", quarter_stays_free},
               {"block_is_carved", block_is_carved},
               {"block_ranges_join", block_ranges_join},
               {"block_and_captures", block_and_captures},
               {"block_given_back_in_a_capture", block_given_back_in_a_capture},
               {"trim_in_a_capture", trim_in_a_capture},
               {"block_yields_to_other_pools", block_yields_to_other_pools},
               {"block_from_threads", block_from_threads}};
  for (auto &t : tests)
    if (argc == 2 && std::string(argv[1]) == t.name) return t.f();
  fprintf(stderr, "unknown test\n");
  return 2;
}
