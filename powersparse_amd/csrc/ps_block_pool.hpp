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
        live_[*ptr] = Live{it->first, device};
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
    live_[*ptr] = Live{bytes, device};
    return Driver::kOk;
  }

  Error Free(void* ptr) {
    Live block{};
    {
      std::lock_guard<std::mutex> lock(mu_);
      const auto it = live_.find(ptr);
      if (it != live_.end()) {
        block = it->second;
        live_.erase(it);
      }
    }
    if (block.bytes == 0) return Driver::Free(ptr);  // a small block
    int current = 0;
    Error e = Driver::Device(&current);
    if (e != Driver::kOk) return e;
    if (current != block.device) e = Driver::SetDevice(block.device);
    if (e != Driver::kOk) return e;
    e = Driver::Synchronize();
    if (e != Driver::kOk) {
      (void)Driver::Free(ptr);
    } else {
      {
        std::lock_guard<std::mutex> lock(mu_);
        Shelf& s = shelves_[block.device];
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
          s.bytes -= it->first;
          it = s.kept.erase(it);
        } else {
          ++it;
        }
      }
      while (s.bytes > s.limit) {
        auto oldest = s.kept.begin();
        for (auto it = s.kept.begin(); it != s.kept.end(); ++it)
          if (it->second.since < oldest->second.since) oldest = it;
        out.push_back(oldest->second.ptr);
        s.bytes -= oldest->first;
        s.kept.erase(oldest);
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
  struct Live {
    size_t bytes;
    int device;
  };
  struct Kept {
    void* ptr;
    int64_t since;
  };
  struct Shelf {
    std::multimap<size_t, Kept> kept;  // by size
    size_t bytes = 0, limit = 0;
  };

  // The driver's allocation; the kept blocks may be what is missing.
  Error DriverMalloc(void** ptr, size_t bytes) {
    Error e = Driver::Malloc(ptr, bytes);
    if (e != Driver::kOutOfMemory) return e;
    Driver::ClearError();
    int device = 0;
    e = Driver::Device(&device);
    if (e == Driver::kOk) e = Trim(device, true);
    return e == Driver::kOk ? Driver::Malloc(ptr, bytes) : e;
  }

  std::mutex mu_;
  std::unordered_map<void*, Live> live_;
  std::map<int, Shelf> shelves_;  // per device
};

}  // namespace ps
