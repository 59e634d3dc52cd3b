// Pipelined host-to-device upload (see staged_upload.h).
#include "staged_upload.h"

#include <algorithm>
#include <cstring>
#include <mutex>

#include "matrix_utils.h"

#ifdef _OPENMP
#include <omp.h>
#endif

namespace PowerSparse {
namespace {

// Bytes per DMA, and the copies from which the large chunks are used. Plain
// copies stay below kMinStaged only: the runtime page-locks the caller's memory
// for larger ones, which stalled uploads of 2 to 4 MB for 3.8 to 4.8 ms (a 10 k-
// node build 2.7 -> 2.2 ms, a first one 6.7 -> 2.5; C1 36.6 -> 35.2 ms).
constexpr size_t kLargeChunk = size_t(32) << 20, kLargeCopy = size_t(64) << 20;
constexpr size_t kSmallChunk = size_t(4) << 20;
constexpr size_t kMinStaged = size_t(64) << 10;
constexpr size_t kCopyBlock = size_t(1) << 20;    // host-copy work item
// Host threads filling a staging buffer: the copy is bound by host memory
// bandwidth, and 8 threads beat 16 (measured on the MI355X box: 103 vs 84 GB/s
// into page-locked memory; C3 upload 33 -> 26 ms, the DMA engine's 56 GB/s
// being the limit).
constexpr int kCopyThreads = 8;

// Two page-locked buffers shared by every upload of the process of one of the
// two chunk sizes (allocated on first use, kept until exit); one upload at a
// time uses them.
struct StagingPool {
  explicit StagingPool(size_t bytes) : chunk(bytes) {}
  const size_t chunk;
  std::mutex mu;
  void* buf[2] = {nullptr, nullptr};
  bool tried = false;
};

StagingPool& Pool(bool large) {
  // never destroyed: they outlive every upload
  static StagingPool* const pools[2] = {new StagingPool(kSmallChunk),
                                        new StagingPool(kLargeChunk)};
  return *pools[large ? 1 : 0];
}

void ParallelCopy(void* dst, const void* src, size_t bytes) {
  const long long blocks = (long long)((bytes + kCopyBlock - 1) / kCopyBlock);
  if (blocks == 1) {  // no team for one block
    std::memcpy(dst, src, bytes);
    return;
  }
#ifdef _OPENMP
  const int threads = std::max(1, std::min(kCopyThreads, omp_get_max_threads()));
#endif
#pragma omp parallel for schedule(static) num_threads(threads)
  for (long long b = 0; b < blocks; ++b) {
    const size_t off = size_t(b) * kCopyBlock;
    std::memcpy(static_cast<char*>(dst) + off, static_cast<const char*>(src) + off,
                std::min(kCopyBlock, bytes - off));
  }
}

// Waits for the stream on scope exit, so that no DMA still reads a staging
// buffer when the pool is released (also on an error path).
struct DrainOnExit {
  ps_stream_t stream;
  ~DrainOnExit() { (void)ps_stream_synchronize(stream); }
};

struct Events {
  ps_event_t e[2] = {nullptr, nullptr};
  ~Events() {
    for (ps_event_t x : e)
      if (x) (void)ps_event_destroy(x);
  }
};

}  // namespace

void StagedUpload(void* dst, const void* src, size_t bytes) {
  if (bytes < kMinStaged) {
    ThrowOnError(ps_memcpy_htod(dst, src, bytes));
    return;
  }
  StagingPool& pool = Pool(bytes >= kLargeCopy);
  const size_t chunk = pool.chunk;
  std::lock_guard<std::mutex> lock(pool.mu);
  if (!pool.tried) {
    pool.tried = true;
    for (void*& b : pool.buf) {
      if (ps_host_malloc(&b, chunk) != PS_OK) b = nullptr;
    }
  }
  if (!pool.buf[0] || !pool.buf[1]) {  // no page-locked memory: plain copy
    ThrowOnError(ps_memcpy_htod(dst, src, bytes));
    return;
  }
  Events ev;
  for (ps_event_t& x : ev.e) ThrowOnError(ps_event_create(&x));
  ps_stream_t const stream = nullptr;
  DrainOnExit drain{stream};
  const char* s = static_cast<const char*>(src);
  char* d = static_cast<char*>(dst);
  size_t k = 0;
  for (size_t off = 0; off < bytes; off += chunk, ++k) {
    const int b = int(k & 1);
    const size_t len = std::min(chunk, bytes - off);
    if (k >= 2) ThrowOnError(ps_event_synchronize(ev.e[b]));  // buffer b's DMA is done
    ParallelCopy(pool.buf[b], s + off, len);
    ThrowOnError(ps_memcpy_htod_async(d + off, pool.buf[b], len, stream));
    ThrowOnError(ps_event_record(ev.e[b], stream));
  }
  ThrowOnError(ps_stream_synchronize(stream));
}

}  // namespace PowerSparse
