// Builds matrices over and over from several threads with the host library's
// sources on a stand-in runtime, for the sanitizers: the block pool, the
// page-locked staging buffers, the signature-bit thread beside the values'
// upload, the lifetimes of the stages, and the ways out by an exception.
//
// The null stream is a thread that runs what was queued, so copies overlap the
// host as they do on a device. The stages whose results the host reads are
// computed plainly; the others (defined elsewhere, returning 0) do nothing, and
// the gather checks that the uploaded arrays have arrived whole.
#include <atomic>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <limits>
#include <mutex>
#include <random>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

#include "matrix_utils.h"
#include "ps_block_pool.hpp"

namespace {

// ---------------------------------------------------------------- runtime

struct Queue {
  std::mutex mu;
  std::condition_variable more, less;
  std::deque<std::function<void()>> work;
  uint64_t queued = 0, done = 0;
  bool stop = false;
  std::thread worker{[this] { Run(); }};

  void Run() {
    std::unique_lock<std::mutex> lock(mu);
    while (true) {
      more.wait(lock, [this] { return stop || !work.empty(); });
      if (work.empty()) return;
      const std::function<void()> f = std::move(work.front());
      work.pop_front();
      lock.unlock();
      f();
      lock.lock();
      ++done;
      less.notify_all();
    }
  }
  uint64_t Put(std::function<void()> f) {
    std::lock_guard<std::mutex> lock(mu);
    work.push_back(std::move(f));
    more.notify_one();
    return ++queued;
  }
  void Wait(uint64_t until) {
    std::unique_lock<std::mutex> lock(mu);
    less.wait(lock, [&] { return done >= until; });
  }
  void Drain() {
    uint64_t until;
    {
      std::lock_guard<std::mutex> lock(mu);
      until = queued;
    }
    Wait(until);
  }
  ~Queue() {
    {
      std::lock_guard<std::mutex> lock(mu);
      stop = true;
    }
    more.notify_one();
    worker.join();
  }
};
Queue& queue() {
  static Queue q;
  return q;
}

struct Driver {
  using Error = int;
  static constexpr Error kOk = 0, kOutOfMemory = 2, kInvalid = 1;
  static int64_t NowNs() {
    return std::chrono::steady_clock::now().time_since_epoch() / std::chrono::nanoseconds(1);
  }
  static Error Device(int* d) {
    *d = 0;
    return kOk;
  }
  static Error SetDevice(int) { return kOk; }
  static Error Malloc(void** p, size_t n) {
    *p = std::malloc(n);
    return *p ? kOk : kOutOfMemory;
  }
  static Error Free(void* p) {
    std::free(p);
    return kOk;
  }
  static Error Synchronize() {
    queue().Drain();
    return kOk;
  }
  static Error TotalBytes(size_t* t) {
    *t = size_t(2) << 30;
    return kOk;
  }
  static void ClearError() {}
};
ps::BlockPool<Driver>& pool() {
  static ps::BlockPool<Driver> p;
  return p;
}
bool pooled = true;  // else every block goes straight to free, for the sanitizer to see

struct Event {
  std::atomic<uint64_t> at{0};
};
thread_local std::string error;
std::atomic<long long> live_blocks{0};

// what the matrix of this thread is built from
thread_local const int* want_col = nullptr;
thread_local const float* want_val = nullptr;
thread_local size_t want_nnz = 0;
std::atomic<int> gathers{0}, wrong{0};

int Split(long long d, int S, int fine, long long* groups) {
  if (S == 1) {
    groups[0] += (d + fine - 1) / fine;
    return 0;
  }
  for (int s = S - 1; s > 0; --s) {
    const long long n = d / (32LL << (s - 1));
    groups[s] += n;
    d -= n * (32LL << (s - 1));
  }
  groups[0] += d > 0;
  return 0;
}

}  // namespace

extern "C" {
const char* ps_last_error(void) { return error.c_str(); }
int ps_get_device(int* d) { return Driver::Device(d); }
int ps_get_device_props(int, ps_device_props* p) {
  std::memset(p, 0, sizeof(*p));
  p->cu_count = 1;
  return PS_OK;
}
int ps_device_synchronize(void) {
  queue().Drain();
  pool().GiveBackIdle();
  return PS_OK;
}
int ps_malloc(void** p, size_t n) {
  *p = nullptr;
  if (n == 0) return PS_OK;
  ++live_blocks;
  return pooled ? pool().Malloc(p, n) : Driver::Malloc(p, n);
}
int ps_free(void* p) {
  if (!p) return PS_OK;
  --live_blocks;
  if (pooled) return pool().Free(p);
  queue().Drain();
  return Driver::Free(p);
}
int ps_mem_kept(size_t* n) {
  *n = pool().KeptBytes(0);
  return PS_OK;
}
int ps_mem_trim_to(size_t n) { return pool().Trim(0, n); }
int ps_host_malloc(void** p, size_t n) { return Driver::Malloc(p, n); }
int ps_memcpy_htod_async(void* d, const void* s, size_t n, ps_stream_t) {
  if (n == 0) return PS_OK;
  queue().Put([=] { std::memcpy(d, s, n); });
  return PS_OK;
}
int ps_memcpy_dtod_async(void* d, const void* s, size_t n, ps_stream_t) {
  return ps_memcpy_htod_async(d, s, n, nullptr);
}
int ps_memcpy_htod(void* d, const void* s, size_t n) {
  if (n == 0) return PS_OK;
  queue().Wait(queue().Put([=] { std::memcpy(d, s, n); }));
  return PS_OK;
}
int ps_memcpy_dtoh(void* d, const void* s, size_t n) { return ps_memcpy_htod(d, s, n); }
int ps_memset_async(void* d, int v, size_t n, ps_stream_t) {
  if (n == 0) return PS_OK;
  queue().Put([=] { std::memset(d, v, n); });
  return PS_OK;
}
int ps_stream_synchronize(ps_stream_t) {
  queue().Drain();
  return PS_OK;
}
int ps_event_create(ps_event_t* e) {
  *e = reinterpret_cast<ps_event_t>(new Event);
  return PS_OK;
}
int ps_event_destroy(ps_event_t e) {
  delete reinterpret_cast<Event*>(e);
  return PS_OK;
}
int ps_event_record(ps_event_t e, ps_stream_t) {
  reinterpret_cast<Event*>(e)->at = queue().Put([] {});
  return PS_OK;
}
int ps_event_synchronize(ps_event_t e) {
  queue().Wait(reinterpret_cast<Event*>(e)->at);
  return PS_OK;
}

int ps_pre_degree_sums(const int* rp, int rows, unsigned long long* sums, ps_stream_t) {
  queue().Drain();
  std::fill(sums, sums + 32, 0ull);
  for (int r = 0; r < rows; ++r)
    for (int s = 1; s < 26; ++s) sums[s] += unsigned(rp[r + 1] - rp[r]) / (32u << (s - 1));
  return PS_OK;
}
int ps_pre_check_csr(const int* ci, const float* v, int n, int cols, uint32_t* flag, int* bad,
                     ps_stream_t) {
  queue().Drain();
  *bad = 0;
  *flag = 0;
  for (int p = 0; p < n; ++p) {
    if (ci) *bad |= ci[p] < 0 || ci[p] >= cols;
    if (v) *bad |= !(v[p] - v[p] == 0.f);
  }
  return PS_OK;
}
int ps_pre_col_histogram_cols(const int* ci, int nnz, int, int* count, ps_stream_t) {
  queue().Drain();
  for (int p = 0; p < nnz; ++p) ++count[ci[p]];
  return PS_OK;
}
int ps_pre_group_prefix(const int* rp, int rows, int S, int fine, uint32_t*, uint32_t* totals,
                        ps_stream_t) {
  queue().Drain();
  std::vector<long long> groups(size_t(S), 0);
  for (int r = 0; r < rows; ++r) Split(rp[r + 1] - rp[r], S, fine, groups.data());
  for (int s = 0; s < S; ++s) totals[s] = uint32_t(groups[size_t(s)]);
  return PS_OK;
}
int ps_pre_rank_sort(const int*, int, const int* ci, int, const int*, int, int, uint64_t*,
                     uint32_t*, ps_stream_t) {
  queue().Drain();
  if (std::memcmp(ci, want_col, want_nnz * 4)) ++wrong;
  return PS_OK;
}
int ps_pre_gather_workset_cols(int, int, const uint32_t*, int, const int*, const int*,
                               const uint32_t*, const int* ci, const float* v, int*, float*, int*,
                               ps_stream_t) {
  queue().Drain();
  ++gathers;
  if (std::memcmp(ci, want_col, want_nnz * 4) || std::memcmp(v, want_val, want_nnz * 4)) ++wrong;
  return PS_OK;
}
int ps_exclusive_scan_u32(const uint32_t* in, uint32_t* out, size_t n, void*, ps_stream_t) {
  queue().Drain();
  uint32_t run = 0;
  for (size_t i = 0; i < n; ++i) {
    const uint32_t v = in[i];
    out[i] = run;
    run += v;
  }
  return PS_OK;
}
size_t ps_hub_stored_words(const ps_hub_block* hb) { return size_t(hb->rows) * size_t((hb->cols + 31) / 32); }
size_t ps_hub_dense_floats(int rows, int cols) { return size_t(rows) * size_t(cols); }
int ps_hub_select(const int* rp, const int* count, int n, long long lo, long long hi, int* index,
                  int* list, int* selected, ps_stream_t) {
  queue().Drain();
  *selected = 0;
  for (int i = 0; i < n; ++i) {
    const long long v = rp ? rp[i + 1] - rp[i] : count[i];
    index[i] = -1;
    if (v >= lo && v < hi) {
      index[i] = *selected;
      list[(*selected)++] = i;
    }
  }
  return PS_OK;
}
int ps_hub_rest_counts(int, const ps_hub_block* hubs, const int* rp, uint32_t* counts, ps_stream_t) {
  queue().Drain();
  for (int r = 0; r < hubs->matrix_rows; ++r)
    counts[r] = uint32_t(hubs->hub_index[r] < 0 ? rp[r + 1] - rp[r] : (rp[r + 1] - rp[r]) / 2);
  return PS_OK;
}
int ps_hub_tiles(const ps_hub_block*, int, const ps_workset*, uint8_t*, uint32_t*, uint32_t* listed,
                 ps_stream_t) {
  *listed = 0;
  return PS_OK;
}
}

namespace {

struct Csr {
  int rows, cols;
  std::vector<int> rp, ci;
  std::vector<float> v;
};
Csr Make(int rows, int cols, int mean, unsigned seed) {
  std::mt19937 rng(seed);
  Csr a{rows, cols, {0}, {}, {}};
  for (int r = 0; r < rows; ++r) {
    const int d = r < 400 ? mean * 20 : int(rng() % unsigned(2 * mean + 1));
    a.rp.push_back(a.rp.back() + d);
  }
  a.ci.resize(size_t(a.rp.back()));
  a.v.resize(a.ci.size());
  for (int& c : a.ci) c = int(rng() % unsigned(cols)) / (1 + int(rng() % 8));
  for (float& x : a.v) x = float(rng() % 1000) * 1e-3f;
  return a;
}

void BuildOnce(const Csr& a, int kind) {
  using namespace PowerSparse;
  want_col = a.ci.data();
  want_val = a.v.data();
  want_nnz = a.ci.size();
  PartitionPolicy policy;
  policy.csr_positions = kind & 1;
  policy.task_order = kind % 3 == 1 ? TaskOrder::kRow : kind % 3 == 2 ? TaskOrder::kAuto : TaskOrder::kSignature;
  if (kind % 3 == 0 && kind % 2 == 0) {
    policy.hub_min_degree[0] = 256;
    policy.hub_min_count[0] = 4;
  }
  PreprocessTimings t;
  PowerSparseMatrixGPU m(a.rows, a.cols, int(a.ci.size()), a.rp.data(), a.ci.data(), a.v.data(),
                         policy, kind & 2 ? &t : nullptr);
  if (m.MatrixNNZ() != int(want_nnz)) ++wrong;
}

}  // namespace

int main(int argc, char** argv) {
  if (argc != 5) return 2;
  pooled = std::strcmp(argv[1], "pool") == 0;
  const int threads = std::atoi(argv[2]), rounds = std::atoi(argv[3]);
  const bool large = std::strcmp(argv[4], "large") == 0;
  // large: past the size from which the entries are checked on the device
  std::vector<Csr> graphs;
  for (int t = 0; t < threads; ++t)
    graphs.push_back(large ? Make(300000, 150000, 60, unsigned(t) + 1u)
                           : Make(9000, 150000, 24, unsigned(t) + 1u));
  std::vector<std::thread> all;
  for (int t = 0; t < threads; ++t)
    all.emplace_back([&, t] {
      Csr& a = graphs[size_t(t)];
      for (int k = 0; k < rounds; ++k) {
        BuildOnce(a, k + t);
        // the exceptions: a column and a value that the checks find
        for (int e = 0; e < 2; ++e) {
          const size_t at = a.ci.size() - 1;
          const int c = a.ci[at];
          const float x = a.v[at];
          if (e == 0) a.ci[at] = a.cols;
          else a.v[at] = std::numeric_limits<float>::infinity();
          try {
            BuildOnce(a, k);
            ++wrong;
          } catch (const std::invalid_argument&) {
          }
          a.ci[at] = c;
          a.v[at] = x;
          if (large) break;
        }
      }
    });
  for (std::thread& t : all) t.join();
  (void)pool().Trim(0, 0);
  std::printf("%d threads, %d rounds, %zu nonzeros: %d gathers, %d wrong, %lld blocks left\n", threads,
              rounds, graphs[0].ci.size(), gathers.load(), wrong.load(), live_blocks.load());
  return wrong.load() || live_blocks.load() ? 1 : 0;
}
