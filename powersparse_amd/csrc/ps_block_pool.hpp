// Freed device blocks of 2 MB and more, kept for the next allocation.
//
// Building a matrix allocates and frees several times its size, and the driver
// clears the pages it hands out: a program that builds matrix after matrix is
// served from cleared pages for some tens of GB and then waits (32 GB freed in
// 366 - 958 ms, about 33 GB/s; a 264 M-nonzero build slowed from 0.29 s to 0.6 -
// 1.3 s, and a 50 M-nonzero matrix took 8 ms to destroy). A kept block needs
// neither the clearing nor the unmapping.
//
// A block is synchronised with its whole device before it is kept (as hipFree
// does), so any stream or thread may get it next. Sizes are rounded up to 2 MB;
// a kept block serves requests from four fifths of its size up, so an array
// may hold up to a quarter more than was asked for.
//
// What is kept is given back to the driver, oldest first, beyond a sixteenth of
// the device's memory; all of it when an allocation fails; and every block that
// has lain unused for kKeepNs, at the next Malloc or Free of any size or
// GiveBackIdle, which the device-wide synchronisation calls. No thread or timer of
// its own does it (hipFree waits for the device, and is refused while a stream
// is captured), so a program that makes none of these calls keeps its blocks:
// the builder of a matrix trims what the build left (Trim).
//
// The driver's calls come in as a policy, so that the pool compiles without a
// GPU runtime (and is tested there):
//   Error, kOk, kOutOfMemory, kInvalid; NowNs(), Device(int*), SetDevice(int),
//   Malloc(void**, size_t), Free(void*), Synchronize(), TotalBytes(size_t*),
//   ClearError().
#pragma once

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstdint>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace ps {

template <class Driver>
class BlockPool {
 public:
  using Error = typename Driver::Error;
  static constexpr size_t kMin = size_t(2) << 20;
  static constexpr int64_t kKeepNs = int64_t(10) * 1000000000;

  Error Malloc(void** ptr, size_t bytes) {
    const Error e = Take(ptr, bytes);  // (an idle block may be what fits)
    GiveBackIdle();
    return e;
  }

  // kInvalid for a block that is kept already (or being kept by another
  // thread): the driver, which still counts it as allocated, would free it
  // under the pool.
  Error Free(void* ptr) {
    const Error e = Return(ptr);
    GiveBackIdle();
    return e;
  }

  // Gives back the device's kept blocks, oldest first, until at most `keep`
  // bytes are left. A block that the driver will not free stays kept.
  Error Trim(int device, size_t keep) {
    std::vector<Out> out;
    {
      std::lock_guard<std::mutex> lock(mu_);
      Shelf& s = shelves_[device];
      while (s.bytes > keep) {
        auto oldest = s.kept.begin();
        for (auto it = s.kept.begin(); it != s.kept.end(); ++it)
          if (it->second.since < oldest->second.since) oldest = it;
        TakeOut(s, oldest, device, &out);
      }
    }
    return GiveBack(out);
  }

  // Gives back the blocks unused for kKeepNs, on every device. What the driver
  // refuses now is tried again when it has lain as long once more.
  void GiveBackIdle() {
    if (due_.load(std::memory_order_relaxed) == kNever) return;
    const int64_t now = Driver::NowNs();
    if (now < due_.load(std::memory_order_relaxed)) return;
    std::vector<Out> out;
    {
      std::lock_guard<std::mutex> lock(mu_);
      int64_t due = kNever;
      for (auto& shelf : shelves_) {
        Shelf& s = shelf.second;
        for (auto it = s.kept.begin(); it != s.kept.end();) {
          const int64_t at = it->second.since + kKeepNs;
          if (at <= now) {
            it = TakeOut(s, it, shelf.first, &out);
          } else {
            due = std::min(due, at);
            ++it;
          }
        }
      }
      due_ = due;
    }
    if (GiveBack(out) != Driver::kOk) Driver::ClearError();
  }

  // Bytes kept on the device.
  size_t KeptBytes(int device) {
    std::lock_guard<std::mutex> lock(mu_);
    return shelves_[device].bytes;
  }

 private:
  static constexpr int64_t kNever = INT64_MAX;
  // kReturning: in Free, not yet kept.
  enum State { kLive, kReturning, kKept };
  struct Block {
    size_t bytes;
    int device;
    State state;
  };
  struct Kept {
    void* ptr;
    int64_t since;
  };
  struct Shelf {
    std::multimap<size_t, Kept> kept;  // by size
    size_t bytes = 0, limit = 0;
  };
  using KeptAt = typename std::multimap<size_t, Kept>::iterator;
  struct Out {
    void* ptr;
    size_t bytes;
    int device;
  };

  Error Take(void** ptr, size_t bytes) {
    // (what cannot be rounded up is the driver's to refuse)
    if (bytes < kMin || bytes > SIZE_MAX - kMin) return DriverMalloc(ptr, bytes);
    int device = 0;
    Error e = Driver::Device(&device);
    if (e != Driver::kOk) return e;
    bytes = (bytes + kMin - 1) / kMin * kMin;
    {
      std::lock_guard<std::mutex> lock(mu_);
      Shelf& s = shelves_[device];
      const auto it = s.kept.lower_bound(bytes);
      if (it != s.kept.end() && it->first <= bytes + bytes / 4) {
        *ptr = it->second.ptr;
        blocks_[*ptr].state = kLive;
        s.bytes -= it->first;
        s.kept.erase(it);
        return Driver::kOk;
      }
      if (s.limit == 0) {
        size_t total = 0;
        e = Driver::TotalBytes(&total);
        if (e != Driver::kOk) return e;
        s.limit = total / 16;
      }
    }
    e = DriverMalloc(ptr, bytes);
    if (e != Driver::kOk) return e;
    std::lock_guard<std::mutex> lock(mu_);
    blocks_[*ptr] = Block{bytes, device, kLive};
    return Driver::kOk;
  }

  Error Return(void* ptr) {
    Block block{};
    {
      std::lock_guard<std::mutex> lock(mu_);
      const auto it = blocks_.find(ptr);
      if (it != blocks_.end()) {
        if (it->second.state != kLive) return Driver::kInvalid;
        it->second.state = kReturning;
        block = it->second;
      }
    }
    if (block.bytes == 0) return Driver::Free(ptr);  // a small block
    int current = block.device;
    Error e = Driver::Device(&current);
    if (e == Driver::kOk && current != block.device) e = Driver::SetDevice(block.device);
    if (e == Driver::kOk) e = Driver::Synchronize();
    if (e != Driver::kOk) {
      {
        std::lock_guard<std::mutex> lock(mu_);
        blocks_.erase(ptr);
      }
      (void)Driver::Free(ptr);
    } else {
      size_t limit = 0;
      {
        std::lock_guard<std::mutex> lock(mu_);
        Keep(Out{ptr, block.bytes, block.device});
        limit = shelves_[block.device].limit;
      }
      e = Trim(block.device, limit);
    }
    if (current != block.device) {
      const Error back = Driver::SetDevice(current);
      if (e == Driver::kOk) e = back;
    }
    return e;
  }

  // (under the lock)
  void Keep(const Out& o) {
    Shelf& s = shelves_[o.device];
    const int64_t now = Driver::NowNs();
    blocks_[o.ptr] = Block{o.bytes, o.device, kKept};
    s.kept.insert({o.bytes, Kept{o.ptr, now}});
    s.bytes += o.bytes;
    due_ = std::min(due_.load(), now + kKeepNs);
  }
  KeptAt Unlist(Shelf& s, KeptAt it) {
    blocks_.erase(it->second.ptr);
    s.bytes -= it->first;
    return s.kept.erase(it);
  }
  KeptAt TakeOut(Shelf& s, KeptAt it, int device, std::vector<Out>* out) {
    out->push_back(Out{it->second.ptr, it->first, device});
    return Unlist(s, it);
  }

  Error GiveBack(const std::vector<Out>& out) {
    Error first = Driver::kOk;
    for (const Out& o : out) {
      const Error e = Driver::Free(o.ptr);
      if (e == Driver::kOk) continue;
      if (first == Driver::kOk) first = e;
      std::lock_guard<std::mutex> lock(mu_);
      Keep(o);
    }
    return first;
  }

  // The driver's allocation; the kept blocks may be what is missing. An address
  // that the pool still lists was freed behind its back, and is dropped.
  Error DriverMalloc(void** ptr, size_t bytes) {
    Error e = Driver::Malloc(ptr, bytes);
    if (e == Driver::kOutOfMemory) {
      Driver::ClearError();
      int device = 0;
      e = Driver::Device(&device);
      if (e == Driver::kOk) e = Trim(device, 0);
      if (e == Driver::kOk) e = Driver::Malloc(ptr, bytes);
    }
    if (e != Driver::kOk) {
      Driver::ClearError();  // the caller has it; the next launch's check is not for it
      return e;
    }
    std::lock_guard<std::mutex> lock(mu_);
    const auto it = blocks_.find(*ptr);
    if (it == blocks_.end()) return e;
    Shelf& s = shelves_[it->second.device];
    const auto same = s.kept.equal_range(it->second.bytes);
    for (auto k = same.first; k != same.second; ++k)
      if (k->second.ptr == *ptr) {
        Unlist(s, k);
        return e;
      }
    blocks_.erase(it);
    return e;
  }

  std::mutex mu_;
  std::unordered_map<void*, Block> blocks_;
  std::map<int, Shelf> shelves_;  // per device
  std::atomic<int64_t> due_{kNever};  // when the first kept block has lain too long
};

}  // namespace ps
