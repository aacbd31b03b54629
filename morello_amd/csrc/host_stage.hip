// Host buffers to the GPU and back (host_stage.h).
#include "host_stage.h"

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <new>
#include <thread>

namespace mrl {
namespace {

typedef unsigned v4u __attribute__((ext_vector_type(4)));

// `vecs` 16-byte vectors across PCIe, either way (no Spec's kernel: it is in no plan).  16 workgroups keep the link full (55 GB/s; 256 of
// them reach 50: the link wants long runs more than many requests).  The last workgroup to finish
// resets the counter and raises the flag on the host.
constexpr int COPY_BLOCKS = 16;
__global__ __launch_bounds__(256) void pcie_copy(const v4u *__restrict__ src, v4u *__restrict__ dst, uint32_t vecs, uint32_t *counter,
                                                   uint32_t *flag, uint32_t ticket) {
  const uint32_t step = gridDim.x * 256;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < vecs; i += step * 4) {
    v4u v[4];
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (i + u * step < vecs) v[u] = src[i + u * step];
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (i + u * step < vecs) dst[i + u * step] = v[u];
  }
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x != 0) return;
  if (__hip_atomic_fetch_add(counter, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1 != gridDim.x) return;
  __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(flag, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Helper threads for memcpy, started at the first large transfer and then asleep between transfers
// for the life of the process.  One job at a time; others who want the helpers meanwhile do their
// copies alone, as does a process that may have no more threads (it is asked again at the next transfer).
class Helpers {
 public:
  static constexpr int COUNT = 3;
  // Runs f(0) .. f(n - 1), each once, on the caller and the helpers; returns when all are done.
  void run(int n, const std::function<void(int)> &f) {
    if (n < 2 || !busy_.try_lock()) {
      for (int i = 0; i < n; i++) f(i);
      return;
    }
    std::lock_guard<std::mutex> one_job(busy_, std::adopt_lock);
    {
      std::lock_guard<std::mutex> lock(m_);
      try {
        for (; started_ < COUNT; started_++) std::thread([this] { work(); }).detach();
      } catch (const std::exception &) {   // (this is called from C)
      }
      f_ = &f, n_ = n, next_ = 0, inside_ = started_, job_++;
    }
    wake_.notify_all();
    for (int i; (i = next_.fetch_add(1)) < n;) f(i);
    std::unique_lock<std::mutex> lock(m_);
    idle_.wait(lock, [&] { return inside_ == 0; });
  }

 private:
  void work() {
    uint64_t seen = 0;
    for (;;) {
      const std::function<void(int)> *f;
      int n;
      {
        std::unique_lock<std::mutex> lock(m_);
        wake_.wait(lock, [&] { return job_ != seen; });
        seen = job_, f = f_, n = n_;
      }
      for (int i; (i = next_.fetch_add(1)) < n;) (*f)(i);
      std::lock_guard<std::mutex> lock(m_);
      if (--inside_ == 0) idle_.notify_one();
    }
  }
  std::mutex busy_, m_;
  std::condition_variable wake_, idle_;
  int started_ = 0;
  const std::function<void(int)> *f_ = nullptr;
  int n_ = 0, inside_ = 0;
  uint64_t job_ = 0;
  std::atomic<int> next_{0};
};
Helpers &helpers() {
  static Helpers *h = new Helpers;  // never destroyed: its threads sleep on it until the process ends
  return *h;
}

std::mutex g_idle_mutex;
HostStage *g_idle[HostStage::IDLE_MAX];   // the first g_n_idle
int g_n_idle = 0;
void (*g_stream_end)(hipStream_t) = nullptr;

size_t round_up(size_t n, size_t to) { return (n + to - 1) / to * to; }

}  // namespace

void on_host_stage_stream_end(void (*f)(hipStream_t)) { g_stream_end = f; }

hipError_t device_malloc(void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipErrorOutOfMemory && HostStage::drop_idle()) {
    (void)hipGetLastError();   // (the first try's)
    e = hipMalloc(p, bytes);
  }
  return e;
}

hipError_t HostStage::init() {
  hipError_t e = hipGetDevice(&device_id_);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&side_, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&join_, hipEventDisableTiming);
  if (e == hipSuccess) e = hipHostMalloc(reinterpret_cast<void **>(&pin_), PINNED_BYTES, hipHostMallocDefault);
  if (e == hipSuccess) e = hipHostMalloc(reinterpret_cast<void **>(&flags_), SLOTS * 64, hipHostMallocDefault);
  if (e == hipSuccess) e = device_malloc(reinterpret_cast<void **>(&counters_), SLOTS * 64);
  if (e != hipSuccess) return e;
  std::memset(flags_, 0, SLOTS * 64);
  return hipMemset(counters_, 0, SLOTS * 64);
}

HostStage::~HostStage() {
  if (side_) (void)hipStreamSynchronize(side_);
  if (stream_) {
    (void)hipStreamSynchronize(stream_);
    if (g_stream_end) g_stream_end(stream_);
    (void)hipStreamDestroy(stream_);
  }
  if (side_) (void)hipStreamDestroy(side_);
  if (join_) (void)hipEventDestroy(join_);
  if (dev_) (void)hipFree(dev_);
  if (counters_) (void)hipFree(counters_);
  if (pin_) (void)hipHostFree(pin_);
  if (flags_) (void)hipHostFree(flags_);
}

HostStage *HostStage::acquire(size_t bytes, hipError_t *err) {
  int device = 0;
  if ((*err = hipGetDevice(&device)) != hipSuccess) return nullptr;
  HostStage *stage = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_idle_mutex);
    for (int i = 0; i < g_n_idle && !stage; i++)
      if (g_idle[i]->device_id_ == device) stage = g_idle[i], g_idle[i] = g_idle[--g_n_idle];
  }
  if (!stage) {
    stage = new (std::nothrow) HostStage;
    if (!stage) {
      *err = hipErrorOutOfMemory;
      return nullptr;
    }
    if ((*err = stage->init()) != hipSuccess) {
      delete stage;
      return nullptr;
    }
  }
  if (stage->dev_size_ < bytes) {
    if (stage->dev_) (void)hipFree(stage->dev_);
    stage->dev_ = nullptr, stage->dev_size_ = 0;
    const size_t want = round_up(bytes, size_t(2) << 20);
    *err = device_malloc(reinterpret_cast<void **>(&stage->dev_), want);
    if (*err == hipErrorOutOfMemory && g_stream_end) {   // the scratch that earlier calls left on this stage's own stream
      (void)hipGetLastError();
      g_stream_end(stage->stream_);
      *err = hipMalloc(reinterpret_cast<void **>(&stage->dev_), want);
    }
    if (*err != hipSuccess) {
      stage->dev_ = nullptr;
      delete stage;
      return nullptr;
    }
    stage->dev_size_ = want;
  }
  *err = hipSuccess;
  return stage;
}

void HostStage::release(HostStage *stage, bool good) {
  if (!good) {
    delete stage;   // waits for what its streams still hold
    return;
  }
  if (stage->dev_size_ > KEEP_DEVICE_BYTES) {
    (void)hipFree(stage->dev_);
    stage->dev_ = nullptr, stage->dev_size_ = 0;
  }
  {
    std::lock_guard<std::mutex> lock(g_idle_mutex);
    if (g_n_idle < IDLE_MAX) {
      g_idle[g_n_idle++] = stage;
      return;
    }
  }
  delete stage;
}

bool HostStage::drop_idle() {
  int device = 0;
  const bool known = hipGetDevice(&device) == hipSuccess;
  bool any = false;
  for (;;) {
    HostStage *s = nullptr;
    {
      std::lock_guard<std::mutex> lock(g_idle_mutex);
      if (g_n_idle > 0) s = g_idle[--g_n_idle];
    }
    if (!s) break;
    (void)hipSetDevice(s->device_id_);
    delete s;
    any = true;
  }
  if (known && any) (void)hipSetDevice(device);
  return any;
}

hipError_t HostStage::copy(void *dst, const void *src, size_t bytes, uint32_t slot, uint32_t ticket, hipStream_t stream) {
  const uint32_t vecs = uint32_t((bytes + 15) / 16);   // both sides are padded to 256 bytes
  const uint32_t blocks = std::min<uint32_t>(COPY_BLOCKS, (vecs + 255) / 256);
  pcie_copy<<<dim3(blocks), dim3(256), 0, stream>>>(static_cast<const v4u *>(src), static_cast<v4u *>(dst), vecs, counters_ + slot * 16,
                                                       flags_ + slot * 16, ticket);
  return hipGetLastError();
}

// Until copy `ticket` of `slot` is complete, or `failed` says that it never will be: by polling the flag,
// then, for work that takes longer, yielding, then asleep in the runtime (which also reports a
// stream that failed).
hipError_t HostStage::wait(uint32_t slot, uint32_t ticket, const std::atomic<int> &failed) {
  const std::atomic<uint32_t> *flag = reinterpret_cast<const std::atomic<uint32_t> *>(flags_ + slot * 16);
  const auto began = std::chrono::steady_clock::now();
  for (uint32_t spin = 1; flag->load(std::memory_order_acquire) != ticket; spin++) {
    if (spin % 256 != 0) {
      __builtin_ia32_pause();
      continue;
    }
    if (failed.load() != int(hipSuccess)) return hipError_t(failed.load());
    const auto waited = std::chrono::steady_clock::now() - began;
    if (waited > std::chrono::milliseconds(5)) {
      hipError_t e = hipStreamSynchronize(stream_);
      if (e == hipSuccess) e = hipStreamSynchronize(side_);
      if (e != hipSuccess) return e;
    }
    if (waited > std::chrono::microseconds(200)) sched_yield();
  }
  return hipSuccess;
}

// The stage's bytes from the first piece to the last, cut into parts, so that the host's copies and the
// link's overlap.  P parts cost P launches of 3 us and leave the last part's trip over the link
// (total / P / 55 GB/s) uncovered: least at a part of sqrt(total * 165 KB).  At most PART_MAX.
struct HostStage::Parts {
  const Piece *pieces;
  int n_pieces;
  size_t first, total, part;
  int count;
  Parts(const Piece *p, int n) : pieces(p), n_pieces(n), first(p[0].offset), total(p[n - 1].offset + p[n - 1].bytes - p[0].offset) {
    part = std::min(PART_MAX, round_up(size_t(std::sqrt(double(total) * 165e3)), 4096));
    count = int((total + part - 1) / part);
  }
  size_t from(int i) const { return size_t(i) * part; }
  size_t bytes(int i) const { return std::min(total - from(i), part); }
  // Between a part's slot and what of each piece falls into the part.
  void host_copy(int i, uint8_t *slot, bool in) const {
    for (int p = 0; p < n_pieces; p++) {
      const size_t p0 = pieces[p].offset - first, p1 = p0 + pieces[p].bytes;
      const size_t lo = std::max(from(i), p0), hi = std::min(from(i) + bytes(i), p1);
      if (lo >= hi) continue;
      uint8_t *host = static_cast<uint8_t *>(pieces[p].host) + (lo - p0), *pinned = slot + (lo - from(i));
      if (in) std::memcpy(pinned, host, hi - lo);
      else std::memcpy(host, pinned, hi - lo);
    }
  }
  // Transfers of megabytes are worth waking the helpers for (a wake-up takes as long as half a
  // megabyte's copy).
  template <class F>
  void for_each(F &&f) const {
    if (total >= (size_t(2) << 20)) helpers().run(count, std::ref(f));   // (a reference: nothing to allocate)
    else for (int i = 0; i < count; i++) f(i);
  }
  // From four parts on every second one takes the stage's other stream: a copy then starts while the
  // one before it drains (launch gap and PCIe round trip, ~5 us of a part's 37).
  bool two_streams() const { return count >= 4; }
};

hipError_t HostStage::upload(const Piece *pieces, int n) {
  if (n == 0) return hipSuccess;
  const Parts parts(pieces, n);
  std::atomic<int> failed{int(hipSuccess)};
  const uint32_t ticket = ticket_ + 1;
  ticket_ += uint32_t((parts.count + SLOTS - 1) / SLOTS);
  // Part i goes through slot i % SLOTS once part i - SLOTS has left it (parts are taken in order, so
  // whoever has that one is ahead).
  auto one = [&](int i) {
    const uint32_t slot = uint32_t(i % SLOTS), round = uint32_t(i / SLOTS);
    hipError_t e = hipSetDevice(device_id_);
    if (e == hipSuccess && round > 0) e = wait(slot, ticket + round - 1, failed);
    uint8_t *pinned = pin_ + size_t(slot) * PART_MAX;
    if (e == hipSuccess) {
      parts.host_copy(i, pinned, true);
      e = copy(dev_ + parts.first + parts.from(i), pinned, parts.bytes(i), slot, ticket + round, (i & 1) && parts.two_streams() ? side_ : stream_);
    }
    if (e != hipSuccess) failed = int(e);
  };
  parts.for_each(one);
  if (failed.load() != int(hipSuccess) || !parts.two_streams()) return hipError_t(failed.load());
  const hipError_t e = hipEventRecord(join_, side_);
  return e == hipSuccess ? hipStreamWaitEvent(stream_, join_, 0) : e;
}

hipError_t HostStage::download(const Piece *pieces, int n) {
  if (n == 0) return hipStreamSynchronize(stream_);
  const Parts parts(pieces, n);
  std::atomic<int> failed{int(hipSuccess)};
  const uint32_t ticket = ticket_ + 1;
  ticket_ += uint32_t((parts.count + SLOTS - 1) / SLOTS);
  auto fetch = [&](int i) {   // (the slots may still hold an upload: its copies are ahead in the stream)
    const uint32_t slot = uint32_t(i % SLOTS);
    const hipError_t e = copy(pin_ + size_t(slot) * PART_MAX, dev_ + parts.first + parts.from(i), parts.bytes(i), slot, ticket + uint32_t(i / SLOTS),
                              (i & 1) && parts.two_streams() ? side_ : stream_);
    if (e != hipSuccess) failed = int(e);
  };
  if (parts.two_streams()) {
    hipError_t e = hipEventRecord(join_, stream_);
    if (e == hipSuccess) e = hipStreamWaitEvent(side_, join_, 0);
    if (e != hipSuccess) return e;
  }
  for (int i = 0; i < std::min(parts.count, SLOTS); i++) fetch(i);
  auto one = [&](int i) {
    const uint32_t slot = uint32_t(i % SLOTS);
    hipError_t e = hipSetDevice(device_id_);
    if (e == hipSuccess) e = wait(slot, ticket + uint32_t(i / SLOTS), failed);
    if (e == hipSuccess) {
      parts.host_copy(i, pin_ + size_t(slot) * PART_MAX, false);
      if (i + SLOTS < parts.count) fetch(i + SLOTS);
    } else {
      failed = int(e);
    }
  };
  parts.for_each(one);
  return hipError_t(failed.load());
}

}  // namespace mrl
