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
// What is kept is bounded by a sixteenth of the device's memory, oldest given
// back first.
//
// The driver's calls come in as a policy, so that the pool compiles without a
// GPU runtime (and is tested there):
//   Error, kOk, kOutOfMemory, kInvalid; NowNs(), Device(int*), SetDevice(int),
//   Malloc(void**, size_t), Free(void*), Synchronize(), TotalBytes(size_t*),
//   ClearError().
#pragma once

#include <algorithm>
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

  // kInvalid for a block that is kept already (or being kept by another
  // thread): the driver, which still counts it as allocated, would free it
  // under the pool.
  Error Free(void* ptr) {
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
      {
        std::lock_guard<std::mutex> lock(mu_);
        Shelf& s = shelves_[block.device];
        blocks_[ptr].state = kKept;
        s.kept.insert({block.bytes, Kept{ptr, Driver::NowNs()}});
        s.bytes += block.bytes;
      }
      e = Trim(block.device, false);
    }
    if (current != block.device) {
      const Error back = Driver::SetDevice(current);
      if (e == Driver::kOk) e = back;
    }
    return e;
  }

  // Gives back the device's kept blocks: those beyond its limit (oldest first)
  // or unused too long, or with `all` every one.
  Error Trim(int device, bool all) {
    std::vector<void*> out;
    {
      std::lock_guard<std::mutex> lock(mu_);
      Shelf& s = shelves_[device];
      const int64_t old = Driver::NowNs() - kKeepNs;
      for (auto it = s.kept.begin(); it != s.kept.end();) {
        if (all || it->second.since < old) {
          out.push_back(it->second.ptr);
          it = Unlist(s, it);
        } else {
          ++it;
        }
      }
      while (s.bytes > s.limit) {
        auto oldest = s.kept.begin();
        for (auto it = s.kept.begin(); it != s.kept.end(); ++it)
          if (it->second.since < oldest->second.since) oldest = it;
        out.push_back(oldest->second.ptr);
        Unlist(s, oldest);
      }
    }
    for (void* ptr : out) {
      const Error e = Driver::Free(ptr);
      if (e != Driver::kOk) return e;
    }
    return Driver::kOk;
  }

  // Bytes kept on the device.
  size_t KeptBytes(int device) {
    std::lock_guard<std::mutex> lock(mu_);
    return shelves_[device].bytes;
  }

 private:
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

  // (under the lock)
  KeptAt Unlist(Shelf& s, KeptAt it) {
    blocks_.erase(it->second.ptr);
    s.bytes -= it->first;
    return s.kept.erase(it);
  }

  // The driver's allocation; the kept blocks may be what is missing. An address
  // that the pool still lists was freed behind its back, and is dropped.
  Error DriverMalloc(void** ptr, size_t bytes) {
    Error e = Driver::Malloc(ptr, bytes);
    if (e == Driver::kOutOfMemory) {
      Driver::ClearError();
      int device = 0;
      e = Driver::Device(&device);
      if (e == Driver::kOk) e = Trim(device, true);
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
};

}  // namespace ps
