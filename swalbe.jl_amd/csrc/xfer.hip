// xfer.hip -- fields between host arrays and a film's device planes.
//
// A field crosses in chunks through pinned host buffers.  The GPU converts
// (element type, FP32 deviation encoding) while it reads or writes the pinned
// chunk over PCIe, so a field makes one pass over the link and the host only
// copies plain bytes to or from the caller's array; for large fields a few
// threads share that copy and the page faults of a fresh array.
//
// What bounds it: the caller's memory (first touch of its pages) and PCIe
// (56 GB/s with pinned buffers).  Converting on the host instead (a loop with
// one 64-bit division per value over a pageable copy) took 44 ms for the
// height of a 4096 x 4096 FP32 film (67 MB); this takes 4 ms.
#include <string.h>

#include <atomic>
#include <chrono>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <type_traits>
#include <vector>

#include "swalbe_internal.h"

namespace swalbe {

namespace {

constexpr size_t kChunk = (size_t)1 << 19;  // bytes of one pinned buffer
constexpr size_t kKeep = 10;                // idle buffers kept per device while films live
// threads that copy a field of this many bytes: 1, 2 from 4 MB, 4 from 8 MB
// (67 MB into fresh memory: 5.2 ms with one, 1.8 with four, 1.9 with eight;
// a first upload of 2 MB, with its buffers to be allocated, takes 260 us with
// two threads and buffers of 1 MB, 190 with one and 512 KB)
inline int copy_threads(size_t bytes) {
  return bytes >= ((size_t)8 << 20) ? 4 : bytes >= ((size_t)4 << 20) ? 2 : 1;
}

// ---------------------------------------------------------------- pinned buffers
constexpr int kFlags = 16;

struct Stage {
  int device = 0;
  char* pin = nullptr;  // kChunk bytes and the flags behind them
  hipEvent_t ev = nullptr;
  uint32_t seq = 0;  // the flags' value after the buffer's last flagged kernel

  uint32_t* flag() const { return (uint32_t*)(pin + kChunk); }
};

// Waits for a kernel whose n workgroups end by setting a flag of its buffer
// each: polls for up to 100 us, which is quicker by 5 us than waiting for the
// stream, then waits for the stream (which also reports a kernel that failed).
hipError_t flag_wait(const Stage& st, int n, hipStream_t s) {
  const auto t0 = std::chrono::steady_clock::now();
  for (;;) {
    for (int i = 0; i < 64; ++i) {
      while (n > 0 && __atomic_load_n(st.flag() + n - 1, __ATOMIC_ACQUIRE) == st.seq) --n;
      if (n == 0) return hipSuccess;
      __builtin_ia32_pause();
    }
    if (std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(100))
      return hipStreamSynchronize(s);
  }
}

void stage_free(Stage& s) {
  if (s.ev) (void)hipEventDestroy(s.ev);
  if (s.pin) (void)hipHostFree(s.pin);
  s = Stage{};
}

// Buffers of finished transfers, for the next one on the same device.  Held
// only while films (or batches) exist: the last one's destruction frees them.
struct Pool {
  std::mutex mu;
  std::vector<Stage> idle;
  long live = 0;
};
Pool& pool() {
  static Pool* p = new Pool;  // never destroyed: no HIP call after main
  return *p;
}

hipError_t stage_take(int device, Stage* out) {
  {
    Pool& P = pool();
    std::lock_guard<std::mutex> lk(P.mu);
    for (size_t i = P.idle.size(); i-- > 0;)
      if (P.idle[i].device == device) {
        *out = P.idle[i];
        P.idle.erase(P.idle.begin() + (long)i);
        return hipSuccess;
      }
  }
  Stage s;
  s.device = device;
  hipError_t e = hipHostMalloc((void**)&s.pin, kChunk + kFlags * sizeof(uint32_t),
                               hipHostMallocPortable | hipHostMallocCoherent);
  for (int i = 0; e == hipSuccess && i < kFlags; ++i) s.flag()[i] = 0;
  if (e == hipSuccess) e = hipEventCreateWithFlags(&s.ev, hipEventDisableTiming);
  if (e != hipSuccess) {
    stage_free(s);
    return e;
  }
  *out = s;
  return hipSuccess;
}

// The buffer's transfer has completed (its event was waited for).
void stage_give(Stage& s) {
  if (!s.pin) return;
  {
    Pool& P = pool();
    std::lock_guard<std::mutex> lk(P.mu);
    size_t same = 0;
    for (const Stage& t : P.idle) same += t.device == s.device;
    if (P.live > 0 && same < kKeep) {
      try {
        P.idle.push_back(s);
        s = Stage{};
        return;
      } catch (...) {  // no room to remember it: freed below
      }
    }
  }
  stage_free(s);
}

// ---------------------------------------------------------------- kernels
// Host elements [a, b) of a field whose plane k (n elements) lies at
// dev + k * stride; blockIdx.y counts the planes from k0 = a / n.
struct Piece {
  int64_t a, b, n, stride;
  int k0;
};

// plane offsets of the FP32 encoding (one for scalar fields), 0: plain values
struct Offsets {
  double v[kQ];
};

template <typename TD, typename TH, bool BITS>
__global__ __launch_bounds__(256) void k_to_host(const TD* __restrict__ dev, TH* __restrict__ pin,
                                                 Piece P, Offsets off) {
  const int k = P.k0 + (int)blockIdx.y;
  const int64_t lo = P.a > k * P.n ? P.a : k * P.n;
  const int64_t hi = P.b < (k + 1) * P.n ? P.b : (k + 1) * P.n;
  const TD* src = dev + k * (P.stride - P.n);
  const double o = off.v[k];
  for (int64_t i = lo + blockIdx.x * 256 + threadIdx.x; i < hi; i += (int64_t)gridDim.x * 256) {
    if constexpr (BITS) {
      pin[i - P.a] = src[i];
    } else {
      const double v = (double)src[i];
      pin[i - P.a] = (TH)(o == 0.0 ? v : v + o);
    }
  }
}

template <typename TD, typename TH, bool BITS>
__global__ __launch_bounds__(256) void k_from_host(TD* __restrict__ dev,
                                                   const TH* __restrict__ pin, Piece P,
                                                   Offsets off) {
  const int k = P.k0 + (int)blockIdx.y;
  const int64_t lo = P.a > k * P.n ? P.a : k * P.n;
  const int64_t hi = P.b < (k + 1) * P.n ? P.b : (k + 1) * P.n;
  TD* dst = dev + k * (P.stride - P.n);
  const double o = off.v[k];
  for (int64_t i = lo + blockIdx.x * 256 + threadIdx.x; i < hi; i += (int64_t)gridDim.x * 256) {
    if constexpr (BITS) dst[i] = pin[i - P.a];
    else dst[i] = (TD)((double)pin[i - P.a] - o);
  }
}

// FP32 planes re-encoded in place: decoded with the old offset, encoded with
// the new one, in FP64 as a download and an upload would.
__global__ __launch_bounds__(256) void k_reencode(float* __restrict__ dev, int64_t n,
                                                  int64_t stride, Offsets from, Offsets to) {
  float* p = dev + blockIdx.y * stride;
  const double a = from.v[blockIdx.y], b = to.v[blockIdx.y];
  for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const double v = (double)p[i];
    p[i] = (float)((a == 0.0 ? v : v + a) - b);
  }
}

// A small field in a few workgroups, each of which tells the host by a flag
// behind its data.  us, with a wait for the stream / so: doubles 1000 down 14 / 9,
// 8000 down 14.8 / 11.3 (the runtime's copy of pageable memory 12) and up 14.8 /
// 10.8 (11.2), 65536 down 32 / 30 and up 29 / 25.  Four elements a thread one after
// the other took 13.5 for 8000 up, one workgroup more than the stream.
constexpr int64_t kSmall = 1024;  // elements of a workgroup, while there are flags for it
constexpr int64_t kFlagged = 65536;

// ONE: at most one element of a plane for each thread (the loop's code alone
// costs a small transfer 0.6 us)
template <typename TD, typename TH, bool BITS, bool DOWN, bool ONE>
__global__ __launch_bounds__(1024) void k_small(TD* __restrict__ dev, TH* __restrict__ pin,
                                                int planes, int64_t n, int64_t stride,
                                                Offsets off, uint32_t* flag, uint32_t seq) {
  const int64_t first = blockIdx.x * 1024 + threadIdx.x, step = 1024 * (int64_t)gridDim.x;
  for (int k = 0; k < planes; ++k) {
    const double o = off.v[k];
    auto cross = [&](int64_t i) {
      if constexpr (BITS) {
        if constexpr (DOWN) pin[k * n + i] = dev[k * stride + i];
        else dev[k * stride + i] = pin[k * n + i];
      } else if constexpr (DOWN) {
        const double v = (double)dev[k * stride + i];
        pin[k * n + i] = (TH)(o == 0.0 ? v : v + o);
      } else {
        dev[k * stride + i] = (TD)((double)pin[k * n + i] - o);
      }
    };
    if constexpr (ONE) {
      if (first < n) cross(first);
    } else {
#pragma unroll 4
      for (int64_t i = first; i < n; i += step) cross(i);
    }
  }
  // a download: every wave's stores have left before the flag's release, which
  // writes the L2 back for all of them (a fence at workgroup scope waits for
  // none); an upload: its loads are back, and the stream orders the plane's next
  // use behind this kernel
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(flag + blockIdx.x, seq, DOWN ? __ATOMIC_RELEASE : __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

Offsets offsets(const double* off, int planes) {
  Offsets o{};
  for (int k = 0; off && k < planes; ++k) o.v[k] = off[k];
  return o;
}

struct Job {
  bool down;
  char* host;
  size_t hes;
  char* dev;
  size_t des;
  int64_t n, stride, total, per;  // per: host elements of one chunk
  int planes, device;
  Offsets off;
  bool bits;
  int groups;   // > 0: so many workgroups, each with a flag (k_small)
  bool single;  // one chunk: its end is the stream's, no event (0.9 us less of 16)
  // an FP32 film and doubles: converted on the host, which crosses half the
  // bytes (200000 doubles up 80 -> 50 us, 1e6 down 270 -> 189); not one so small
  // that a single workgroup takes it
  bool narrow;
  hipStream_t s;
  std::atomic<int64_t> next{0};
  std::atomic<int> err{0};
  std::atomic<bool> no_pinned{false};
};

template <typename TD, typename TH, bool BITS>
void launch_small(const Job& J, const Stage& st) {
  auto go = [&](auto down, auto one) {
    hipLaunchKernelGGL((k_small<TD, TH, BITS, decltype(down)::value, decltype(one)::value>),
                       dim3(J.groups), dim3(1024), 0, J.s, (TD*)J.dev, (TH*)st.pin, J.planes, J.n,
                       J.stride, J.off, st.flag(), st.seq);
  };
  const bool one = J.n <= 1024 * (int64_t)J.groups;
  if (J.down) one ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
  else one ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
}

template <typename TD, typename TH, bool BITS>
void launch_piece(const Job& J, char* pin, const Piece& P, dim3 grid) {
  if (J.down)
    hipLaunchKernelGGL((k_to_host<TD, TH, BITS>), grid, dim3(256), 0, J.s, (const TD*)J.dev,
                       (TH*)pin, P, J.off);
  else
    hipLaunchKernelGGL((k_from_host<TD, TH, BITS>), grid, dim3(256), 0, J.s, (TD*)J.dev,
                       (const TH*)pin, P, J.off);
}

// f(TD, TH, BITS) as types, for the job's elements
template <typename F>
void with_types(const Job& J, F&& f) {
  if (J.bits) {
    if (J.des == 8) f(uint64_t{}, uint64_t{}, std::true_type{});
    else f(uint32_t{}, uint32_t{}, std::true_type{});
  } else if (J.des == 8) {
    if (J.hes == 8) f(double{}, double{}, std::false_type{});
    else f(double{}, float{}, std::false_type{});
  } else {
    if (J.hes == 8) f(float{}, double{}, std::false_type{});
    else f(float{}, float{}, std::false_type{});
  }
}

hipError_t issue(const Job& J, Stage& st, int64_t a, int64_t b) {
  Piece P{a, b, J.n, J.stride, (int)(a / J.n)};
  const int64_t widest = b - a < J.n ? b - a : J.n;
  const dim3 grid((unsigned)((widest + 255) / 256), (unsigned)((b - 1) / J.n - a / J.n + 1));
  if (J.groups) ++st.seq;
  with_types(J, [&](auto td, auto th, auto bits) {
    using TD = decltype(td);
    using TH = decltype(th);
    if (J.groups && J.narrow) launch_small<uint32_t, uint32_t, true>(J, st);
    else if (J.groups) launch_small<TD, TH, decltype(bits)::value>(J, st);
    else if (J.narrow) launch_piece<uint32_t, uint32_t, true>(J, st.pin, P, grid);
    else launch_piece<TD, TH, decltype(bits)::value>(J, st.pin, P, grid);
  });
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && !J.single) e = hipEventRecord(st.ev, J.s);
  return e;
}

// Elements [a, b) between the host array and `t` in the device's type
// (consecutive planes one behind the other)
template <typename TD, typename TH>
void convert(const Job& J, TD* t, int64_t a, int64_t b) {
  TH* const h = (TH*)J.host;
  for (int64_t lo = a; lo < b;) {
    const int64_t k = lo / J.n, hi = (k + 1) * J.n < b ? (k + 1) * J.n : b;
    const double o = J.off.v[k];
    TD* const u = t - a;
    if (!J.down)
      for (int64_t i = lo; i < hi; ++i) u[i] = (TD)((double)h[i] - o);
    else if (o == 0.0)
      for (int64_t i = lo; i < hi; ++i) h[i] = (TH)u[i];
    else
      for (int64_t i = lo; i < hi; ++i) h[i] = (TH)((double)u[i] + o);
    lo = hi;
  }
}

// Elements [a, b) between the host array and a pinned buffer
void stage_copy(const Job& J, char* pin, int64_t a, int64_t b) {
  char* const h = J.host + (size_t)a * J.hes;
  const size_t bytes = (size_t)(b - a) * J.hes;
  if (J.narrow) convert<float, double>(J, (float*)pin, a, b);
  else if (J.down) memcpy(h, pin, bytes);
  else memcpy(pin, h, bytes);
}

// One copying thread: claims chunks until none is left, two buffers in turn
// (the GPU fills or drains one while the host copies the other).
void run_chunks(Job* pJ) {
  Job& J = *pJ;
  Stage st[2];
  int64_t a[2] = {0, 0}, b[2] = {-1, -1};  // chunk in flight in each buffer (b < 0: none)
  hipError_t e = hipSetDevice(J.device);
  auto finish = [&](int r) {  // wait for buffer r; a download's chunk goes to the caller
    if (b[r] < 0) return;
    const hipError_t w = J.groups   ? flag_wait(st[r], J.groups, J.s)
                         : J.single ? hipStreamSynchronize(J.s)
                                    : hipEventSynchronize(st[r].ev);
    if (w == hipSuccess && J.down && e == hipSuccess)
      stage_copy(J, st[r].pin, a[r], b[r]);
    if (e == hipSuccess) e = w;
    b[r] = -1;
  };
  for (int r = 0; e == hipSuccess && J.err.load() == 0; r ^= 1) {
    const int64_t c = J.next.fetch_add(1);
    if (c * J.per >= J.total) break;
    finish(r);
    if (e == hipSuccess && !st[r].pin) {
      e = stage_take(J.device, &st[r]);
      if (e != hipSuccess) {
        (void)hipGetLastError();
        J.no_pinned.store(true);
      }
    }
    if (e != hipSuccess) break;
    a[r] = c * J.per;
    const int64_t end = a[r] + J.per < J.total ? a[r] + J.per : J.total;
    if (!J.down) stage_copy(J, st[r].pin, a[r], end);
    e = issue(J, st[r], a[r], end);
    if (e == hipSuccess) b[r] = end;
  }
  // the chunk issued last may sit in either buffer: drain both
  finish(0);
  finish(1);
  stage_give(st[0]);
  stage_give(st[1]);
  if (e != hipSuccess) {
    int none = 0;
    J.err.compare_exchange_strong(none, (int)e);
  }
}

// The transfer without pinned memory: the runtime's own copy, converted on the
// host.  (It takes 10 to 40 us for the same 64 KB, as the array happens to lie.)
hipError_t run_plain(const Job& J) {
  hipError_t e = hipSetDevice(J.device);
  if (e != hipSuccess) return e;
  const size_t row = (size_t)J.n * J.des, pitch = (size_t)J.stride * J.des;
  std::unique_ptr<char[]> tmp(J.bits ? nullptr : new (std::nothrow) char[row * J.planes]);
  if (!J.bits && !tmp) return hipErrorOutOfMemory;
  char* h = J.bits ? J.host : tmp.get();
  auto converted = [&] {
    with_types(J, [&](auto td, auto th, auto) {
      convert<decltype(td), decltype(th)>(J, (decltype(td)*)tmp.get(), 0, J.total);
    });
  };
  if (!J.down && !J.bits) converted();
  if (J.planes == 1)
    e = J.down ? hipMemcpyAsync(h, J.dev, row, hipMemcpyDeviceToHost, J.s)
               : hipMemcpyAsync(J.dev, h, row, hipMemcpyHostToDevice, J.s);
  else
    e = J.down ? hipMemcpy2DAsync(h, row, J.dev, pitch, row, J.planes, hipMemcpyDeviceToHost, J.s)
               : hipMemcpy2DAsync(J.dev, pitch, h, row, row, J.planes, hipMemcpyHostToDevice, J.s);
  if (e == hipSuccess) e = hipStreamSynchronize(J.s);
  if (e == hipSuccess && J.down && !J.bits) converted();
  return e;
}

int transfer(bool down, void* host, size_t hes, void* dev, size_t des, int64_t n, int planes,
             int64_t stride, const double* off, int device, hipStream_t s) {
  Job J;
  J.down = down;
  J.host = (char*)host;
  J.hes = hes;
  J.dev = (char*)dev;
  J.des = des;
  J.n = n;
  J.stride = stride;
  J.planes = planes;
  J.total = n * planes;
  J.groups = J.total > kFlagged ? 0 : J.total > kFlags * kSmall ? kFlags : (int)((J.total - 1) / kSmall + 1);
  J.narrow = J.groups != 1 && des < hes;
  J.per = (int64_t)(kChunk / (J.narrow ? des : hes));
  J.single = J.total <= J.per;
  J.device = device;
  J.off = offsets(off, planes);
  J.bits = hes == des;
  for (int k = 0; k < planes; ++k) J.bits = J.bits && J.off.v[k] == 0.0;
  J.s = s;
  std::vector<std::thread> helpers;
  try {
    for (int i = 1; i < copy_threads((size_t)J.total * hes); ++i)
      helpers.emplace_back(run_chunks, &J);
  } catch (...) {  // no further thread: those that run share the chunks
  }
  run_chunks(&J);
  for (std::thread& t : helpers) t.join();
  if (J.no_pinned.load()) J.err.store((int)run_plain(J));
  if (J.err.load() != 0)
    return hip_fail((hipError_t)J.err.load(), down ? "copy to host" : "copy to device");
  return SWALBE_OK;
}

}  // namespace

int field_to_host(void* host, size_t hes, const void* dev, size_t des, int64_t n, int planes,
                  int64_t stride, const double* off, int device, hipStream_t s) {
  return transfer(true, host, hes, const_cast<void*>(dev), des, n, planes, stride, off, device, s);
}

int field_from_host(void* dev, size_t des, const void* host, size_t hes, int64_t n, int planes,
                    int64_t stride, const double* off, int device, hipStream_t s) {
  return transfer(false, const_cast<void*>(host), hes, dev, des, n, planes, stride, off, device,
                  s);
}

void launch_reencode(float* dev, int64_t n, int planes, int64_t stride, const double* from,
                     const double* to, hipStream_t s) {
  const int64_t b = (n + 255) / 256;
  hipLaunchKernelGGL(k_reencode, dim3((unsigned)(b < 65535 ? b : 65535), (unsigned)planes),
                     dim3(256), 0, s, dev, n, stride, offsets(from, planes), offsets(to, planes));
}

HostResult::HostResult(int device, hipStream_t s) : s_(s) {
  Stage* st = new (std::nothrow) Stage;
  if (st && stage_take(device, st) != hipSuccess) (void)hipGetLastError();
  stage_ = st;
  p_ = st ? (double*)st->pin : nullptr;
}

HostResult::~HostResult() {
  Stage* st = (Stage*)stage_;
  if (!st) return;
  // a kernel launched without get() may still write: the buffer goes back when
  // it cannot
  if (st->pin && __atomic_load_n(st->flag(), __ATOMIC_ACQUIRE) != st->seq)
    (void)hipStreamSynchronize(s_);
  stage_give(*st);
  delete st;
}

uint32_t* HostResult::flag() const { return p_ ? ((Stage*)stage_)->flag() : nullptr; }
uint32_t HostResult::seq() { return p_ ? ++((Stage*)stage_)->seq : 0; }

hipError_t HostResult::get(double* out, int n) {
  const hipError_t e = p_ ? flag_wait(*(Stage*)stage_, 1, s_) : hipStreamSynchronize(s_);
  if (e == hipSuccess && p_) memcpy(out, p_, sizeof(double) * (size_t)n);
  return e;
}

void xfer_retain() {
  Pool& P = pool();
  std::lock_guard<std::mutex> lk(P.mu);
  ++P.live;
}

void xfer_release() {
  Pool& P = pool();
  std::vector<Stage> gone;
  {
    std::lock_guard<std::mutex> lk(P.mu);
    if (--P.live == 0) gone.swap(P.idle);
  }
  for (Stage& s : gone) stage_free(s);
}

}  // namespace swalbe
