// Solutions between the device's cell blocks [unit][v][node] and the
// reference layout [unit][node][v] in host memory (uploads and downloads of
// grids, ensembles, adaptive grids and finite-volume patches).
//
// The data take one trip: a kernel reads the blocks and writes the reference
// layout straight into pinned memory (or the other way round), and host
// threads move it between there and the caller's pageable array, whose pages
// are mostly touched there for the first time.  Two buffers alternate, so the
// link and the threads work at the same time.  Before, every chunk was copied
// to a pageable buffer and transposed by one host thread, with the GPU idle:
// the download of 27^3 cells at N = 5 (170 MB) took 33 ms, of 12 x 13 x 14
// patches of 15^3 volumes (295 MB) 90 ms; now 5 and 7 ms.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "host_util.h"

namespace {
constexpr int V = 5;
constexpr size_t CHUNK = 8u << 20;         // bytes of one buffer
constexpr size_t PER_THREAD = 2u << 20;    // a thread more for so many bytes
constexpr int MAX_THREADS = 8;
// A helper polls for its next chunk so long and then sleeps: more than a chunk
// takes on the link (150 us), far less than the steps that a transfer may have
// to wait for.
constexpr std::chrono::microseconds POLL{500};

// words of whole units; UP: reference layout to blocks
template <bool UP>
__global__ __launch_bounds__(256) void k_reorder(double* __restrict__ blocks, double* __restrict__ ref, unsigned words,
                                                 unsigned nodes) {
  const unsigned per = V * nodes;
  for (unsigned i = blockIdx.x * 256u + threadIdx.x; i < words; i += gridDim.x * 256u) {
    const unsigned unit = i / per, e = i - unit * per, node = e / V, v = e - node * V;
    double* b = blocks + (size_t)unit * per + (size_t)v * nodes + node;
    if (UP)
      *b = ref[i];
    else
      ref[i] = *b;
  }
}

// The same through one pageable buffer and the calling thread, where there is
// no pinned memory to be had.
int plain(hipStream_t stream, double* blocks, double* user, long long units, int nodes, bool up) {
  const size_t per = (size_t)V * nodes;
  const long long chunk = std::max<long long>(1, (long long)(CHUNK / (per * sizeof(double))));
  std::vector<double> buf(per * std::min(chunk, units));
  for (long long u0 = 0; u0 < units; u0 += chunk) {
    const long long n = std::min(chunk, units - u0);
    double* ref = user + u0 * per;
    const size_t bytes = sizeof(double) * per * n;
    if (up) {
      for (size_t i = 0; i < per * n; ++i) {
        const size_t e = i % per;
        buf[i - e + e % V * nodes + e / V] = ref[i];
      }
      EXA_CHECK(hipMemcpyAsync(blocks + u0 * per, buf.data(), bytes, hipMemcpyHostToDevice, stream));
    } else {
      EXA_CHECK(hipMemcpyAsync(buf.data(), blocks + u0 * per, bytes, hipMemcpyDeviceToHost, stream));
    }
    EXA_CHECK(hipStreamSynchronize(stream));
    if (!up)
      for (size_t i = 0; i < per * n; ++i) {
        const size_t e = i % per;
        ref[i] = buf[i - e + e % V * nodes + e / V];
      }
  }
  return EXA_OK;
}

// What the threads that share the copying of every chunk know.
class Progress {
  std::atomic<long long> open_{0};  // chunks that may be copied
  std::atomic<bool> stop_{false};
  std::mutex mu_;  // of the changes, for those that sleep
  std::condition_variable changed_;

 public:
  std::atomic<long long> copied{0};  // parts copied by the helpers
  std::atomic<int> parts{1};         // of a chunk; set before the first one opens
  void open(long long chunks) {
    {
      std::lock_guard<std::mutex> lk(mu_);
      open_.store(chunks, std::memory_order_release);
    }
    changed_.notify_all();
  }
  void stop() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_.store(true, std::memory_order_release);
    }
    changed_.notify_all();
  }
  // Waits until chunk k may be copied; false: it will not be.
  bool wait(long long k) {
    auto open = [&] { return open_.load(std::memory_order_acquire) > k; };
    auto stopped = [&] { return stop_.load(std::memory_order_acquire); };
    const auto until = std::chrono::steady_clock::now() + POLL;
    while (!open() && !stopped() && std::chrono::steady_clock::now() < until) std::this_thread::yield();
    if (!open() && !stopped()) {
      std::unique_lock<std::mutex> lk(mu_);
      changed_.wait(lk, [&] { return open() || stopped(); });
    }
    return open();
  }
};
struct Helpers {
  Progress& progress;
  std::vector<std::thread> threads;
  ~Helpers() {
    progress.stop();
    for (auto& t : threads) t.join();
  }
};
}  // namespace

HostStage::~HostStage() {
  for (int i = 0; i < 2; ++i) {
    if (buf[i]) (void)hipHostFree(buf[i]);
    if (ev[i]) (void)hipEventDestroy(ev[i]);
  }
}

bool HostStage::ensure(size_t n) {
  for (int i = 0; i < 2; ++i) {
    if (!ev[i] && hipEventCreateWithFlags(&ev[i], hipEventDisableTiming) != hipSuccess) {
      ev[i] = nullptr;
      (void)hipGetLastError();
      return false;
    }
    if (words >= n) continue;
    if (buf[i]) (void)hipHostFree(buf[i]);
    buf[i] = nullptr;
    void* p = nullptr;
    if (hipHostMalloc(&p, n * sizeof(double), hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      words = 0;
      return false;
    }
    buf[i] = static_cast<double*>(p);
  }
  words = std::max(words, n);
  return true;
}

int exa_transfer_nodes(HostStage& st, hipStream_t stream, double* blocks, double* user, long long units, int nodes,
                       bool up) try {
  if (units <= 0) return EXA_OK;
  std::lock_guard<std::mutex> lk(st.mu);
  const size_t per = (size_t)V * nodes;
  const long long chunk = std::min(units, std::max<long long>(1, (long long)(CHUNK / (per * sizeof(double)))));
  if (!st.ensure(chunk * per)) return plain(stream, blocks, user, units, nodes, up);
  const long long nchunks = (units + chunk - 1) / chunk;
  auto words = [&](long long k) { return (size_t)std::min(chunk, units - k * chunk) * per; };
  const int parts =
      (int)std::min<size_t>(MAX_THREADS, 1 + per * units * sizeof(double) / PER_THREAD);
  Progress pr;
  int nparts = 1;
  auto copy = [&](long long k, int part, int of) {
    const size_t n = words(k), a = n * part / of, b = n * (part + 1) / of;
    double *ref = user + (size_t)k * chunk * per + a, *pin = st.buf[k & 1] + a;
    if (up)
      std::memcpy(pin, ref, (b - a) * sizeof(double));
    else
      std::memcpy(ref, pin, (b - a) * sizeof(double));
  };
  auto help = [&](int part) {
    for (long long k = 0; k < nchunks; ++k) {
      if (!pr.wait(k)) return;
      copy(k, part, pr.parts.load(std::memory_order_relaxed));
      pr.copied.fetch_add(1, std::memory_order_release);
    }
  };
  Helpers helpers{pr, {}};
  helpers.threads.reserve(parts);
  try {
    for (; nparts < parts; ++nparts) helpers.threads.emplace_back(help, nparts);
  } catch (const std::exception&) {  // no more threads: those there are share the work
  }
  pr.parts.store(nparts, std::memory_order_relaxed);
  auto launch = [&](long long k) -> int {
    const unsigned n = (unsigned)words(k);
    const dim3 grid((n + 255) / 256);
    double* b = blocks + (size_t)k * chunk * per;
    if (up)
      hipLaunchKernelGGL(k_reorder<true>, grid, dim3(256), 0, stream, b, st.buf[k & 1], n, (unsigned)nodes);
    else
      hipLaunchKernelGGL(k_reorder<false>, grid, dim3(256), 0, stream, b, st.buf[k & 1], n, (unsigned)nodes);
    EXA_CHECK(hipGetLastError());
    EXA_CHECK(hipEventRecord(st.ev[k & 1], stream));
    return EXA_OK;
  };
  auto share = [&](long long k) {  // copies chunk k with the helpers
    pr.open(k + 1);
    copy(k, 0, nparts);
    while (pr.copied.load(std::memory_order_acquire) < (k + 1) * (nparts - 1)) std::this_thread::yield();
  };
  if (up) {
    for (long long k = 0; k < nchunks; ++k) {
      if (k >= 2) EXA_CHECK(hipEventSynchronize(st.ev[k & 1]));  // the buffer has been read
      share(k);
      EXA_TRY(launch(k));
    }
    EXA_CHECK(hipStreamSynchronize(stream));
    return EXA_OK;
  }
  for (long long k = 0; k < std::min(2LL, nchunks); ++k) EXA_TRY(launch(k));
  for (long long k = 0; k < nchunks; ++k) {
    EXA_CHECK(hipEventSynchronize(st.ev[k & 1]));
    share(k);
    if (k + 2 < nchunks) EXA_TRY(launch(k + 2));
  }
  return EXA_OK;
} catch (const std::exception& e) {
  exa_set_error("moving the solution: %s", e.what());
  return EXA_ERR_NOMEM;
}
