// Checks of the kept-block pool (powersparse_amd/csrc/ps_block_pool.hpp) on a
// stand-in driver: memory of 1 GB per device that is counted, not used, a clock
// that the checks set, and errors for a free of what is not allocated.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "ps_block_pool.hpp"

namespace {

constexpr size_t MB = size_t(1) << 20;

enum Status { kFine = 0, kNoMemory = 2, kBadValue = 1 };

struct Fake {
  using Error = Status;
  static constexpr Error kOk = kFine, kOutOfMemory = kNoMemory, kInvalid = kBadValue;

  static inline std::mutex mu;
  static inline std::map<void*, size_t> allocated;
  static inline size_t in_use = 0, mallocs = 0;
  static inline uintptr_t next = uintptr_t(1) << 40;
  static inline std::atomic<int64_t> now{0};
  static inline bool refuse_free = false;
  static inline bool left = false;  // an error that the next check would report
  static inline uintptr_t again = 0;  // the next allocation's address, if set

  static int64_t NowNs() { return now; }
  static Error Device(int* device) {
    *device = 0;
    return kOk;
  }
  static Error SetDevice(int) { return kOk; }
  static Error Malloc(void** ptr, size_t bytes) {
    std::lock_guard<std::mutex> lock(mu);
    *ptr = nullptr;
    if (bytes == 0) return kOk;
    if (bytes > 1024 * MB - in_use) {
      left = true;
      return kOutOfMemory;
    }
    *ptr = reinterpret_cast<void*>(again ? again : next);
    if (!again) next += (bytes + 4095) / 4096 * 4096;
    again = 0;
    allocated[*ptr] = bytes;
    in_use += bytes;
    ++mallocs;
    return kOk;
  }
  static Error Free(void* ptr) {
    std::lock_guard<std::mutex> lock(mu);
    if (refuse_free) return kBadValue;
    const auto it = allocated.find(ptr);
    if (it == allocated.end()) return kBadValue;
    in_use -= it->second;
    allocated.erase(it);
    return kOk;
  }
  static Error Synchronize() { return kOk; }
  static Error TotalBytes(size_t* total) {
    *total = 1024 * MB;
    return kOk;
  }
  static void ClearError() { left = false; }
};

using Pool = ps::BlockPool<Fake>;

#define CHECK(cond)                                                   \
  do {                                                                \
    if (!(cond)) {                                                    \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #cond);          \
      return 1;                                                       \
    }                                                                 \
  } while (0)

// Sizes whose rounding up to 2 MB does not fit size_t are out of memory.
int huge() {
  Pool pool;
  for (size_t bytes : {size_t(-1), size_t(-1) - 2 * MB + 2, size_t(-1) - 2 * MB, size_t(1) << 63}) {
    void* p = &pool;
    CHECK(pool.Malloc(&p, bytes) == kNoMemory);
    CHECK(p == nullptr);
    CHECK(!Fake::left);
  }
  CHECK(Fake::in_use == 0);
  return 0;
}

// A second free of a kept block is refused, and the block handed out once.
int double_free() {
  Pool pool;
  void *p = nullptr, *a = nullptr, *b = nullptr;
  CHECK(pool.Malloc(&p, 8 * MB) == kFine && pool.Free(p) == kFine);
  CHECK(pool.Free(p) == kBadValue);
  CHECK(Fake::allocated.count(p) == 1);
  CHECK(pool.KeptBytes(0) == 8 * MB);
  CHECK(pool.Malloc(&a, 8 * MB) == kFine && a == p);
  CHECK(pool.Malloc(&b, 8 * MB) == kFine && b != p);
  CHECK(Fake::allocated.count(a) == 1);
  CHECK(pool.Free(a) == kFine && pool.Free(b) == kFine);
  CHECK(pool.Trim(0, 0) == kFine && Fake::in_use == 0);
  CHECK(pool.Free(a) == kBadValue);  // given back: the driver's answer
  return 0;
}

// A block freed behind the pool's back: when the driver hands its address out
// again, the pool knows the new block, not the old one's size.
int freed_elsewhere() {
  Pool pool;
  void *p = nullptr, *q = nullptr;
  CHECK(pool.Malloc(&p, 8 * MB) == kFine);
  CHECK(Fake::Free(p) == kFine);
  Fake::again = reinterpret_cast<uintptr_t>(p);
  CHECK(pool.Malloc(&q, 4096) == kFine && q == p);
  CHECK(pool.Free(q) == kFine);
  CHECK(pool.KeptBytes(0) == 0 && Fake::in_use == 0);
  // the same for a kept one
  CHECK(pool.Malloc(&p, 8 * MB) == kFine && pool.Free(p) == kFine);
  CHECK(Fake::Free(p) == kFine);
  Fake::again = reinterpret_cast<uintptr_t>(p);
  CHECK(pool.Malloc(&q, 4 * MB) == kFine && q == p);
  CHECK(pool.KeptBytes(0) == 0);
  CHECK(pool.Free(q) == kFine && pool.KeptBytes(0) == 4 * MB);
  CHECK(pool.Trim(0, 0) == kFine && Fake::in_use == 0);
  return 0;
}

// Blocks unused for ten seconds go back at the next call of any kind.
int idle() {
  for (int call = 0; call < 4; ++call) {
    Pool pool;
    void *small = nullptr, *live = nullptr, *a = nullptr, *b = nullptr, *p = nullptr;
    CHECK(pool.Malloc(&small, 4096) == kFine && pool.Malloc(&live, 64 * MB) == kFine);
    CHECK(pool.Malloc(&a, 8 * MB) == kFine && pool.Malloc(&b, 16 * MB) == kFine);
    CHECK(pool.Free(a) == kFine);
    Fake::now += Pool::kKeepNs / 2;
    CHECK(pool.Free(b) == kFine && pool.KeptBytes(0) == 24 * MB);
    Fake::now += Pool::kKeepNs / 2;  // the first is due, the second is not
    const size_t in_use = Fake::in_use;
    if (call == 0) pool.GiveBackIdle();
    if (call == 1) CHECK(pool.Malloc(&p, 64) == kFine);
    if (call == 2) CHECK(pool.Free(small) == kFine);
    if (call == 3) CHECK(pool.Free(live) == kFine && pool.Trim(0, 16 * MB) == kFine);
    CHECK(Fake::allocated.count(a) == 0);
    if (call == 3) continue;  // (the freed 64 MB are the newest)
    CHECK(pool.KeptBytes(0) == 16 * MB && Fake::in_use <= in_use - 8 * MB + 64);
    Fake::now += Pool::kKeepNs;
    pool.GiveBackIdle();
    CHECK(pool.KeptBytes(0) == 0);
  }
  return 0;
}

// A kept block that fits is used, however long it has lain.
int idle_reuse() {
  Pool pool;
  void *a = nullptr, *p = nullptr;
  CHECK(pool.Malloc(&a, 8 * MB) == kFine && pool.Free(a) == kFine);
  Fake::now += 3 * Pool::kKeepNs;
  CHECK(pool.Malloc(&p, 8 * MB) == kFine && p == a && Fake::mallocs == 1);
  return 0;
}

// What the driver refuses to free stays kept, and goes later.
int refused() {
  Pool pool;
  void *a = nullptr, *b = nullptr, *p = nullptr;
  CHECK(pool.Malloc(&a, 8 * MB) == kFine && pool.Malloc(&b, 8 * MB) == kFine);
  CHECK(pool.Free(a) == kFine && pool.Free(b) == kFine);
  Fake::refuse_free = true;
  Fake::now += 2 * Pool::kKeepNs;
  pool.GiveBackIdle();
  CHECK(pool.KeptBytes(0) == 16 * MB);
  CHECK(pool.Trim(0, 0) == kBadValue && pool.KeptBytes(0) == 16 * MB);
  Fake::refuse_free = false;
  CHECK(pool.Malloc(&p, 8 * MB) == kFine && (p == a || p == b));
  Fake::now += 2 * Pool::kKeepNs;
  pool.GiveBackIdle();
  CHECK(pool.KeptBytes(0) == 0 && Fake::in_use == 8 * MB);
  return 0;
}

// Trimming to a size: the oldest go first. The bound of a sixteenth likewise.
int trim_to() {
  Pool pool;
  void* p[40];
  for (void*& q : p) CHECK(pool.Malloc(&q, 2 * MB) == kFine);
  for (void* q : p) {
    ++Fake::now;
    CHECK(pool.Free(q) == kFine);
  }
  CHECK(pool.KeptBytes(0) == 64 * MB);
  for (int k = 0; k < 40; ++k) CHECK(Fake::allocated.count(p[k]) == (k < 8 ? 0u : 1u));
  CHECK(pool.Trim(0, 11 * MB) == kFine && pool.KeptBytes(0) == 10 * MB);
  for (int k = 0; k < 40; ++k) CHECK(Fake::allocated.count(p[k]) == (k < 35 ? 0u : 1u));
  CHECK(pool.Trim(0, 11 * MB) == kFine && pool.KeptBytes(0) == 10 * MB);
  return 0;
}

// Threads that allocate, hold and free while another trims: a block belongs to
// one thread at a time, and nothing is lost.
int threads() {
  Pool pool;
  std::mutex mu;
  std::map<void*, int> owner;
  std::atomic<bool> wrong{false};
  auto work = [&](int t) {
    unsigned x = unsigned(t) * 2654435761u + 1u;
    std::vector<void*> mine;
    for (int k = 0; k < 3000; ++k) {
      x = x * 1664525u + 1013904223u;
      if (mine.size() < 4 && (x >> 16) % 2) {
        void* p = nullptr;
        if (pool.Malloc(&p, 4096 + (x >> 8) % (6 * MB)) != kFine) continue;
        std::lock_guard<std::mutex> lock(mu);
        if (!owner.emplace(p, t).second) wrong = true;
        mine.push_back(p);
      } else if (!mine.empty()) {
        void* const p = mine.back();
        mine.pop_back();
        {
          std::lock_guard<std::mutex> lock(mu);
          owner.erase(p);
        }
        if (pool.Free(p) != kFine) wrong = true;
      }
      if (t == 0 && k % 16 == 0) (void)pool.Trim(0, 8 * MB);
      if (t == 1) Fake::now += Pool::kKeepNs / 64;
    }
    for (void* p : mine) {
      {
        std::lock_guard<std::mutex> lock(mu);
        owner.erase(p);
      }
      if (pool.Free(p) != kFine) wrong = true;
    }
  };
  std::vector<std::thread> all;
  for (int t = 0; t < 6; ++t) all.emplace_back(work, t);
  for (std::thread& t : all) t.join();
  CHECK(!wrong);
  CHECK(pool.Trim(0, 0) == kFine && pool.KeptBytes(0) == 0 && Fake::in_use == 0);
  return 0;
}

struct Check {
  const char* name;
  int (*run)();
};
const Check kChecks[] = {{"huge", huge},
                         {"double_free", double_free},
                         {"freed_elsewhere", freed_elsewhere},
                         {"idle", idle},
                         {"idle_reuse", idle_reuse},
                         {"refused", refused},
                         {"trim_to", trim_to},
                         {"threads", threads}};

}  // namespace

int main(int argc, char** argv) {
  for (const Check& c : kChecks)
    if (argc == 2 && std::strcmp(argv[1], c.name) == 0) return c.run();
  return 2;
}
