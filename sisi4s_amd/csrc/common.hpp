// Common infrastructure of the engine: error propagation (no exceptions
// cross the C ABI), device memory pool, strided tensor views.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdint>
#include <cstdio>
#include <map>
#include <mutex>
#include <set>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

#include "../../include/sisi_engine.h"

namespace sisi {

// Internal failures are C++ exceptions carrying a SISI_ERR_* code; the C ABI
// layer converts them into a status and the thread-local message.
struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

void set_last_error(const std::string &msg);

#define SISI_HIP(call)                                                      \
  do {                                                                      \
    hipError_t e_ = (call);                                                 \
    if (e_ != hipSuccess)                                                   \
      throw ::sisi::Error(SISI_ERR_HIP, std::string(#call) + ": " +         \
                                            hipGetErrorString(e_) + " (" + \
                                            __FILE__ + ":" +                \
                                            std::to_string(__LINE__) + ")"); \
  } while (0)

#define SISI_REQUIRE(cond, code, msg)                                       \
  do {                                                                      \
    if (!(cond)) throw ::sisi::Error((code), (msg));                        \
  } while (0)

// Device memory pool: buffers are recycled by exact byte size, so the
// allocation pattern of one CCSD iteration is served without hipMalloc after
// the first iteration.  Buffers up to kSlabMax are carved out of slabs of
// growing size (8 to 256 MB): hipMalloc and hipFree cost 50 to 100 us each
// whatever the size, and a small system's engine holds a few hundred buffers
// (the batch of 16 systems with No about 10, Nv about 70: 433 -> 264 ms, most
// of it the frees at the end).  Not thread-safe (one engine, one host thread).
// Device-wide operations (hipDeviceSynchronize, hipFree, stream creation and
// destruction) are not allowed while another thread captures its stream into
// a hipGraph: they take this process-wide lock, and so does a capture.
inline std::recursive_mutex &device_wide_mutex() {
  static std::recursive_mutex m;
  return m;
}

//
// A pool also holds at most one block: a large buffer whose contents its owner
// can do without (the pair integrals of the ladder, 124 GB at No = 40, Nv =
// 400).  It is there for whoever needs memory.  While it is not lent, the
// pool's own buffers are carved out of it when less than a quarter of the
// device is free; and an allocation that would fail takes the block of its own pool or of another
// pool of the process, lent or not, back to the device (block_lost() then
// tells the owner), except while the owner has work in hand that reads it
// (begin_use() to end_use()).  Carving comes before freeing since pages that
// were freed are wiped at about 33 GB/s before they can be had again: a mixed
// run after an FP64 run at that size waited 3.1 s for them.
class Pool {
 public:
  Pool() {
    std::lock_guard<std::mutex> lock(registry_mutex());
    registry().push_back(this);
  }
  Pool(const Pool &) = delete;
  Pool &operator=(const Pool &) = delete;
  ~Pool() {
    {
      std::lock_guard<std::mutex> lock(registry_mutex());
      auto &r = registry();
      r.erase(std::find(r.begin(), r.end(), this));
    }
    release_all();
  }
  void *get(size_t bytes) {
    if (bytes == 0) bytes = 8;
    bytes = (bytes + 255) & ~size_t(255);
    auto it = free_.find(bytes);
    if (it != free_.end() && !it->second.empty()) {
      void *p = it->second.back();
      it->second.pop_back();
      hold(p, 1);
      live_.insert(p);
      if (capturing_) captured_.insert(p);
      return p;
    }
    if (void *p = carve(bytes)) return handed_out(p, bytes);
    void *p = bytes > kSlabMax && prefer_block(bytes) ? carve_block(bytes) : nullptr;
    if (!p) p = device_malloc(bytes);
    if (!p) p = carve_block(bytes);
    if (!p) {
      // Drop cached buffers and retry, then take blocks.
      trim();
      p = device_malloc(bytes);
      int waits = 0;
      while (!p) {
        bool busy = false;  // a block in use, which may soon be had
        if (!reclaim(busy)) {
          if (!busy || ++waits > kWaits)
            throw Error(SISI_ERR_ALLOC, "device allocation of " +
                                            std::to_string(bytes) + " bytes failed");
          std::this_thread::sleep_for(std::chrono::milliseconds(20));
        }
        p = device_malloc(bytes);
      }
    }
    return handed_out(p, bytes);
  }
  // The block, of `bytes` bytes: the one kept from an earlier use or a new
  // one; null when it cannot be had.  One that fits a slab is a buffer like
  // any other (nobody is short of so little, and 16 small systems took 16
  // times the 100 us of a hipMalloc and its hipFree longer).
  void *take_block(size_t bytes) {
    if (bytes <= kSlabMax) {
      try {
        return small_block_ = get(bytes);
      } catch (const Error &) {
        return nullptr;
      }
    }
    {
      std::lock_guard<std::mutex> lock(block_m_);
      if (block_.base && (block_.lent || !block_.whole())) return nullptr;
      if (block_.base && block_.size >= bytes) {
        block_.lent = true;
        return block_.base;
      }
    }
    free_idle_block();  // too small
    void *p = device_malloc(bytes);
    if (!p) {
      trim();
      p = device_malloc(bytes);
    }
    if (!p) return nullptr;
    std::lock_guard<std::mutex> lock(block_m_);
    block_ = Block();
    block_.base = static_cast<char *>(p);
    block_.size = bytes;
    block_.room[block_.base] = bytes;
    block_.lent = true;
    (void)hipGetDevice(&block_.device);
    return p;
  }
  // Its owner no longer needs what is in it.
  void return_block() {
    put(small_block_);
    small_block_ = nullptr;
    std::lock_guard<std::mutex> lock(block_m_);
    block_.lent = false;
    lost_ = false;
  }
  // Size of the block if it can be had whole.
  size_t idle_block() const {
    std::lock_guard<std::mutex> lock(block_m_);
    return !block_.lent && block_.whole() ? block_.size : 0;
  }
  // Some of the pool's own buffers are carved out of it.
  bool block_carved() const { return !in_block_.empty(); }
  // A lent block was taken by another allocation.
  bool block_lost() const { return lost_; }
  // The owner issues work that reads or writes the block.
  void begin_use() {
    while (busy_.exchange(true)) std::this_thread::yield();  // a reclaim frees it
  }
  void end_use() { busy_ = false; }
  void put(void *p) {
    if (!p) return;
    auto it = size_.find(p);
    if (it == size_.end()) return;
    live_.erase(p);
    if (reserved_.count(p)) return;  // held by a captured graph
    recycle(p);
  }
  // Graph capture: every buffer handed out between begin_capture and
  // end_capture is referenced by the captured graph, so end_capture takes
  // them out of circulation until release() (when the graph is destroyed);
  // a buffer that still has an owner at release() returns to the free list
  // when that owner gives it back.
  void begin_capture() {
    capturing_ = true;
    captured_.clear();
  }
  std::vector<void *> end_capture() {
    capturing_ = false;
    std::vector<void *> held;
    for (void *p : captured_) {
      if (reserved_.count(p)) continue;
      reserved_.insert(p);
      held.push_back(p);
      if (unlist(p)) hold(p, 1);
    }
    captured_.clear();
    // what else of the block was given back in the course of the capture
    const std::set<void *> carved = in_block_;
    for (void *p : carved)
      if (unlist(p)) recycle(p);
    return held;
  }
  void release(const std::vector<void *> &held) {
    for (void *p : held) {
      reserved_.erase(p);
      if (size_.count(p) && !live_.count(p)) recycle(p);
    }
  }
  // Device memory that can be had again: what trim() gives back (the free
  // lists, of slabs those none of whose buffers is in use) and what is free of
  // a block that is not lent.
  size_t cached_bytes() const {
    size_t b = 0;
    for (const auto &kv : free_)
      for (void *p : kv.second)
        if (!slab_of_.count(p) && !in_block_.count(p)) b += kv.first;
    for (const auto &s : slabs_)
      if (s.base && s.held == 0) b += s.size;
    std::lock_guard<std::mutex> lock(block_m_);
    if (block_.base && !block_.lent)
      for (const auto &r : block_.room) b += r.second;
    return b;
  }
  void trim() {
    std::lock_guard<std::recursive_mutex> lock(device_wide_mutex());
    (void)hipDeviceSynchronize();
    // cached buffers, and the slabs none of whose buffers is in use; not those
    // that launches of the capture in progress use
    std::set<size_t> captured;
    for (void *p : captured_)
      if (slab_of_.count(p)) captured.insert(slab_of_[p]);
    auto held = [&](size_t slab) { return slabs_[slab].held > 0 || captured.count(slab); };
    for (auto &kv : free_) {
      std::vector<void *> keep;
      for (void *p : kv.second) {
        auto it = slab_of_.find(p);
        if ((it != slab_of_.end() && held(it->second)) || in_block_.count(p) ||
            captured_.count(p)) {
          keep.push_back(p);
          continue;
        }
        if (it == slab_of_.end()) (void)hipFree(p);
        else slab_of_.erase(it);
        size_.erase(p);
      }
      kv.second.swap(keep);
    }
    for (size_t i = 0; i < slabs_.size(); ++i)
      if (slabs_[i].base && !held(i)) {
        (void)hipFree(slabs_[i].base);
        slabs_[i] = Slab();
      }
    free_idle_block();
  }
  void release_all() {
    std::lock_guard<std::recursive_mutex> lock(device_wide_mutex());
    (void)hipDeviceSynchronize();
    for (auto &kv : size_)
      if (!slab_of_.count(kv.first) && !in_block_.count(kv.first)) (void)hipFree(kv.first);
    for (auto &s : slabs_)
      if (s.base) (void)hipFree(s.base);
    {
      std::lock_guard<std::mutex> block_lock(block_m_);
      if (block_.base) (void)hipFree(block_.base);
      block_ = Block();
    }
    in_block_.clear();
    slabs_.clear();
    slab_of_.clear();
    next_slab_ = kSlabFirst;
    size_.clear();
    free_.clear();
    reserved_.clear();
    live_.clear();
  }

 private:
  static constexpr size_t kSlabMax = size_t(64) << 20;    // largest carved buffer
  static constexpr size_t kSlabFirst = size_t(8) << 20;   // first slab, then doubling
  static constexpr size_t kSlabLast = size_t(256) << 20;  // up to this
  struct Slab {
    char *base = nullptr;
    size_t size = 0, used = 0;
    int held = 0;  // its buffers outside the free lists
  };
  // A buffer from the first slab with room, or from a new one; null when it
  // is too large or no slab can be had.
  void *carve(size_t bytes) {
    if (bytes > kSlabMax) return nullptr;
    size_t i = 0;
    while (i < slabs_.size() && (!slabs_[i].base || slabs_[i].size - slabs_[i].used < bytes)) ++i;
    if (i == slabs_.size()) {
      Slab s;
      s.size = std::max(next_slab_, 2 * bytes);
      void *p = nullptr;
      if (hipMalloc(&p, s.size) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
      }
      s.base = static_cast<char *>(p);
      slabs_.push_back(s);
      next_slab_ = std::min(2 * next_slab_, kSlabLast);
    }
    Slab &s = slabs_[i];
    void *p = s.base + s.used;
    s.used += bytes;
    slab_of_[p] = i;
    hold(p, 1);
    return p;
  }
  void hold(void *p, int d) {
    auto it = slab_of_.find(p);
    if (it != slab_of_.end()) slabs_[it->second].held += d;
  }
  // A buffer nobody owns: into its free list, or back into the block (in the
  // course of a capture into the list: end_capture() reserves it there).
  void recycle(void *p) {
    if (in_block_.count(p) && !capturing_) {
      std::lock_guard<std::mutex> lock(block_m_);
      block_.give(static_cast<char *>(p), size_[p]);
      in_block_.erase(p);
      size_.erase(p);
      return;
    }
    free_[size_[p]].push_back(p);
    hold(p, -1);
  }
  // Takes a buffer out of its free list; false when it is not in it.
  bool unlist(void *p) {
    auto &fl = free_[size_[p]];
    auto it = std::find(fl.begin(), fl.end(), p);
    if (it == fl.end()) return false;
    fl.erase(it);
    return true;
  }
  static void *device_malloc(size_t bytes) {
    void *p = nullptr;
    if (hipMalloc(&p, bytes) == hipSuccess) return p;
    (void)hipGetLastError();
    return nullptr;
  }
  struct Block {
    char *base = nullptr;
    size_t size = 0;
    int device = 0;
    bool lent = false;
    std::map<char *, size_t> room;  // free ranges, none next to another
    bool whole() const { return base && room.size() == 1 && room.begin()->second == size; }
    // the smallest range that holds n bytes
    char *take(size_t n) {
      auto best = room.end();
      for (auto it = room.begin(); it != room.end(); ++it)
        if (it->second >= n && (best == room.end() || it->second < best->second)) best = it;
      if (best == room.end()) return nullptr;
      char *p = best->first;
      const size_t rest = best->second - n;
      room.erase(best);
      if (rest > 0) room[p + n] = rest;
      return p;
    }
    void give(char *p, size_t n) {
      auto it = room.emplace(p, n).first;
      auto next = std::next(it);
      if (next != room.end() && p + n == next->first) {
        it->second += next->second;
        room.erase(next);
      }
      if (it != room.begin()) {
        auto prev = std::prev(it);
        if (prev->first + prev->second == p) {
          prev->second += it->second;
          room.erase(it);
        }
      }
    }
  };
  static constexpr int kWaits = 50;  // of 20 ms, for blocks in use
  static std::mutex &registry_mutex() {
    static std::mutex m;
    return m;
  }
  static std::vector<Pool *> &registry() {
    static auto *r = new std::vector<Pool *>;  // outlives every pool
    return *r;
  }
  // A quarter of the device stays free for others while there is an idle
  // block; once it has come to that the block is asked first.
  bool prefer_block(size_t bytes) {
    {
      std::lock_guard<std::mutex> lock(block_m_);
      if (!block_.base || block_.lent) return block_first_ = false;
    }
    size_t free_b = 0, total_b = 0;
    if (!block_first_ && !capturing_)
      block_first_ = hipMemGetInfo(&free_b, &total_b) == hipSuccess && free_b < bytes + total_b / 4;
    return block_first_;
  }
  void *carve_block(size_t bytes) {
    std::lock_guard<std::mutex> lock(block_m_);
    if (!block_.base || block_.lent) return nullptr;
    void *p = block_.take(bytes);
    if (p) in_block_.insert(p);
    return p;
  }
  void free_idle_block() {
    std::lock_guard<std::recursive_mutex> device_lock(device_wide_mutex());
    std::lock_guard<std::mutex> lock(block_m_);
    if (block_.lent || !block_.whole()) return;
    (void)hipDeviceSynchronize();
    (void)hipFree(block_.base);
    block_ = Block();
  }
  // Frees the block if nothing is carved out of it; by a thread that holds
  // busy_ (so that its owner is not using it) and the device-wide lock.
  bool surrender(int device) {
    std::lock_guard<std::mutex> lock(block_m_);
    if (!block_.whole() || block_.device != device) return false;
    (void)hipDeviceSynchronize();
    (void)hipFree(block_.base);
    lost_ = block_.lent;
    block_ = Block();
    return true;
  }
  // One block of this pool or another is freed.  busy: another's is in use.
  bool reclaim(bool &busy) {
    if (capturing_) return false;
    int device = 0;
    (void)hipGetDevice(&device);
    std::lock_guard<std::recursive_mutex> device_lock(device_wide_mutex());
    std::lock_guard<std::mutex> lock(registry_mutex());
    auto attempt = [&](Pool *q) {
      if (q->busy_.exchange(true)) {
        busy = busy || (q != this && q->block_in_use(device));
        return false;
      }
      const bool freed = q->surrender(device);
      q->busy_ = false;
      return freed;
    };
    if (attempt(this)) return true;
    for (Pool *q : registry())
      if (q != this && attempt(q)) return true;
    return false;
  }
  bool block_in_use(int device) {
    std::lock_guard<std::mutex> lock(block_m_);
    return block_.base && block_.lent && block_.device == device;
  }
  void *handed_out(void *p, size_t bytes) {
    size_[p] = bytes;
    live_.insert(p);
    if (capturing_) captured_.insert(p);
    return p;
  }
  mutable std::mutex block_m_;     // block_: another pool may take it
  Block block_;
  std::set<void *> in_block_;      // buffers carved out of it
  std::atomic<bool> busy_{false};  // in use by its owner, or about to be freed
  std::atomic<bool> lost_{false};
  bool block_first_ = false;
  void *small_block_ = nullptr;
  std::vector<Slab> slabs_;
  std::map<void *, size_t> slab_of_;
  size_t next_slab_ = kSlabFirst;
  std::map<size_t, std::vector<void *>> free_;
  std::map<void *, size_t> size_;
  std::set<void *> reserved_;
  std::set<void *> live_;  // handed out and not yet given back
  std::set<void *> captured_;
  bool capturing_ = false;
};

// Owning device buffer of doubles, returned to the pool on destruction.
class DBuf {
 public:
  DBuf() = default;
  DBuf(Pool *pool, size_t n) : pool_(pool), n_(n) {
    p_ = static_cast<double *>(pool->get(n * sizeof(double)));
  }
  DBuf(const DBuf &) = delete;
  DBuf &operator=(const DBuf &) = delete;
  DBuf(DBuf &&o) noexcept { swap(o); }
  DBuf &operator=(DBuf &&o) noexcept {
    reset();
    swap(o);
    return *this;
  }
  ~DBuf() { reset(); }
  void reset() {
    if (pool_ && p_) pool_->put(p_);
    p_ = nullptr;
    n_ = 0;
  }
  double *get() const { return p_; }
  size_t size() const { return n_; }

 private:
  void swap(DBuf &o) {
    std::swap(pool_, o.pool_);
    std::swap(p_, o.p_);
    std::swap(n_, o.n_);
  }
  Pool *pool_ = nullptr;
  double *p_ = nullptr;
  size_t n_ = 0;
};

constexpr int kMaxOrder = 6;

// Strided view of a real tensor: element (x0..x_{order-1}) lives at
// p[sum_k x_k * stride[k]].  Dense tensors have stride[0] = 1 and
// stride[k] = stride[k-1] * len[k-1] (first index fastest).
struct View {
  double *p = nullptr;
  int order = 0;
  int64_t len[kMaxOrder] = {0};
  int64_t stride[kMaxOrder] = {0};

  int64_t size() const {
    int64_t n = 1;
    for (int k = 0; k < order; ++k) n *= len[k];
    return n;
  }
};

inline View dense(double *p, std::initializer_list<int64_t> lens) {
  View v;
  v.p = p;
  v.order = 0;
  int64_t s = 1;
  for (int64_t l : lens) {
    v.len[v.order] = l;
    v.stride[v.order] = s;
    s *= l;
    v.order++;
  }
  return v;
}

// View with explicit strides (element x at p[sum_k x_k * strides_k]).
inline View dense_strided(double *p, std::initializer_list<int64_t> lens,
                          std::initializer_list<int64_t> strides) {
  View v;
  v.p = p;
  v.order = 0;
  auto s = strides.begin();
  for (int64_t l : lens) {
    v.len[v.order] = l;
    v.stride[v.order] = *s++;
    v.order++;
  }
  return v;
}

// Sub-block [lo_k, hi_k) of a view (same order).
inline View subview(const View &v, std::initializer_list<int64_t> lo,
                    std::initializer_list<int64_t> hi) {
  View r = v;
  int k = 0;
  auto l = lo.begin();
  auto h = hi.begin();
  for (; k < v.order; ++k, ++l, ++h) {
    r.p += (*l) * v.stride[k];
    r.len[k] = (*h) - (*l);
  }
  return r;
}

}  // namespace sisi
