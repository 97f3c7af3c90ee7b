// Host-side helpers shared by the C-ABI translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <mutex>

#include "common.h"

#define EXA_ARG(cond, msg)                        \
  do {                                            \
    if (!(cond)) {                                \
      exa_set_error("invalid argument: %s", msg); \
      return EXA_ERR_ARG;                         \
    }                                             \
  } while (0)

#define EXA_TRY(expr)              \
  do {                             \
    int r__ = (expr);              \
    if (r__ != EXA_OK) return r__; \
  } while (0)

// Device buffer that grows on demand and frees itself.  Move-only: a copy
// would free the same allocation twice.
struct DevBuf {
  void* p = nullptr;
  size_t n = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  DevBuf(DevBuf&& o) noexcept : p(o.p), n(o.n) {
    o.p = nullptr;
    o.n = 0;
  }
  DevBuf& operator=(DevBuf&& o) noexcept {
    if (this != &o) {
      if (p) (void)hipFree(p);
      p = o.p;
      n = o.n;
      o.p = nullptr;
      o.n = 0;
    }
    return *this;
  }
  void swap(DevBuf& o) noexcept {
    void* tp = p;
    size_t tn = n;
    p = o.p;
    n = o.n;
    o.p = tp;
    o.n = tn;
  }
  int ensure(size_t bytes) {
    if (bytes <= n) return EXA_OK;
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
    EXA_CHECK(hipMalloc(&p, bytes));
    n = bytes;
    return EXA_OK;
  }
  template <typename T>
  T* as() const { return static_cast<T*>(p); }
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
};

// Two pinned buffers and their events, kept by the object whose solution they
// move (at most 8 MB each, or one cell block), allocated by its first transfer
// and kept for the next ones: up to 16 MB of pinned memory an object.
// One transfer at a time: host threads that move parts of one object take
// their turns (the members of an ensemble share its buffers).
struct HostStage {
  std::mutex mu;  // held by exa_transfer_nodes
  double* buf[2] = {nullptr, nullptr};
  hipEvent_t ev[2] = {nullptr, nullptr};
  size_t words = 0;  // of each buffer
  HostStage() = default;
  HostStage(const HostStage&) = delete;
  HostStage& operator=(const HostStage&) = delete;
  ~HostStage();
  bool ensure(size_t n);  // false: no memory
};
// units blocks [v][node] on the device from (up) or to user's [node][v] in
// host memory, behind the work queued on the stream; complete on return.
int exa_transfer_nodes(HostStage& st, hipStream_t stream, double* blocks, double* user, long long units, int nodes,
                       bool up);

// Sum of a sweep counter (EXA_SWEEP_SLOTS words), cleared if asked for; waits
// for the stream.
static inline int exa_read_sweeps(unsigned long long* count, bool clear, hipStream_t stream, long long* total) {
  unsigned long long h[EXA_SWEEP_SLOTS * EXA_SWEEP_STRIDE];
  EXA_CHECK(hipMemcpyAsync(h, count, sizeof(h), hipMemcpyDeviceToHost, stream));
  EXA_CHECK(hipStreamSynchronize(stream));
  *total = 0;
  for (int i = 0; i < EXA_SWEEP_SLOTS; ++i) *total += (long long)h[i * EXA_SWEEP_STRIDE];
  if (!clear) return EXA_OK;
  EXA_CHECK(hipMemsetAsync(count, 0, sizeof(h), stream));
  EXA_CHECK(hipStreamSynchronize(stream));
  return EXA_OK;
}

static inline unsigned long long exa_big_bits() {
  const double big = 1.0e300;
  unsigned long long b;
  __builtin_memcpy(&b, &big, sizeof(b));
  return b;
}

// A stable time step that is 0 (or not a finite positive number) means a cell
// held NaN entries or a negative pressure: the kernels' dt reduction maps
// every such candidate to 0 so that it wins the global minimum.
static inline int exa_check_dt(double dt, const char* what) {
  if (dt > 0.0 && dt <= 1.7976931348623157e308) return EXA_OK;
  exa_set_error("%s: the stable time step is %g -- the state holds non-finite values or a negative pressure", what,
                dt);
  return EXA_ERR_NUMERICS;
}

// Takes the device address of the allocation-free AMR staging area on the
// current device (amr_capi.hip); called by exa_init once per device.
int exa_amr_noalloc_setup(int dev);
