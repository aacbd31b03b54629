// Host check of morello_amd/csrc/host_stage.hip where the machine runs short: of device memory, of threads.
// Linked against the stand-ins below in place of the HIP runtime: "device" memory is host memory out of a
// budget, the copy kernel a memcpy, everything complete as soon as it is enqueued.
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "../morello_amd/csrc/host_stage.h"

static std::mutex g_mutex;
static std::map<void *, size_t> g_blocks;
static size_t g_budget = size_t(1) << 40, g_used = 0;
static bool g_no_threads = false;

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  std::lock_guard<std::mutex> lock(g_mutex);
  *p = nullptr;
  if (n > g_budget - g_used) return hipErrorOutOfMemory;
  *p = std::aligned_alloc(256, (n + 255) / 256 * 256);
  g_blocks[*p] = n, g_used += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> lock(g_mutex);
  if (!g_blocks.count(p)) return hipErrorInvalidValue;
  g_used -= g_blocks[p], g_blocks.erase(p), std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = std::aligned_alloc(256, (n + 255) / 256 * 256), hipSuccess; }
hipError_t hipHostFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { return std::memset(p, v, n), hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = reinterpret_cast<hipStream_t>(std::malloc(1)), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return std::free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = reinterpret_cast<hipEvent_t>(std::malloc(1)), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return std::free(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
void **__hipRegisterFatBinary(const void *) { static void *handle; return &handle; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipUnregisterFatBinary(void **) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream) {
  return *grid = dim3(1), *block = dim3(1), *lds = 0, *stream = nullptr, hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **args, size_t, hipStream_t) {   // pcie_copy(src, dst, vecs, counter, flag, ticket)
  std::memcpy(*static_cast<void **>(args[1]), *static_cast<void **>(args[0]), size_t(*static_cast<uint32_t *>(args[2])) * 16);
  __atomic_store_n(*static_cast<uint32_t **>(args[4]), *static_cast<uint32_t *>(args[5]), __ATOMIC_RELEASE);
  return hipSuccess;
}
int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *x) {
  typedef int (*real_t)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
  static const real_t real = reinterpret_cast<real_t>(dlsym(RTLD_NEXT, "pthread_create"));
  return g_no_threads ? EAGAIN : real(t, a, f, x);
}
}

using mrl::HostStage;
static constexpr size_t MB = size_t(1) << 20;

static void expect(bool ok, const char *what) {
  if (ok) return;
  std::printf("failed: %s\n", what);
  std::exit(1);
}

// In and out through a stage; every byte has to come back.
static void round_trip(HostStage *stage, size_t bytes) {
  std::vector<uint8_t> in(bytes), out(bytes, 0);
  for (size_t i = 0; i < bytes; i++) in[i] = uint8_t(i * 2654435761u >> 13);
  HostStage::Piece p{in.data(), 0, bytes}, q{out.data(), 0, bytes};
  expect(stage->upload(&p, 1) == hipSuccess && stage->download(&q, 1) == hipSuccess, "round trip");
  expect(in == out, "bytes of a round trip");
}

// A scratch arena kept for a stream, as the library keeps them.
static std::map<hipStream_t, void *> g_arenas;
static void drop_arena(hipStream_t s) {
  if (!g_arenas.count(s)) return;
  (void)hipFree(g_arenas[s]);
  g_arenas.erase(s);
}

int main() {
  hipError_t e;
  mrl::on_host_stage_stream_end(drop_arena);
  // No helper threads to be had, then some.
  g_no_threads = true;
  HostStage *a = HostStage::acquire(9 * MB, &e);
  expect(a, "a stage");
  round_trip(a, 9 * MB);
  g_no_threads = false;
  round_trip(a, 9 * MB);
  round_trip(a, 3 * MB + 5);
  HostStage::release(a, true);
  // What two idle stages and their scratch hold is there for a call that needs it ...
  HostStage *s[2] = {HostStage::acquire(20 * MB, &e), HostStage::acquire(20 * MB, &e)};
  for (HostStage *x : s) {
    expect(x, "two stages");
    expect(hipMalloc(&g_arenas[x->stream()], 30 * MB) == hipSuccess, "scratch");
  }
  for (HostStage *x : s) HostStage::release(x, true);
  expect(g_used > 100 * MB, "idle stages keep their memory");
  g_budget = 110 * MB;
  HostStage *big = HostStage::acquire(100 * MB, &e);
  expect(big, "a stage as large as the device, idle ones given back");
  round_trip(big, 100 * MB);
  HostStage::release(big, true);
  // ... and for any other allocation of the library.
  void *p = nullptr;
  expect(mrl::device_malloc(&p, 105 * MB) == hipSuccess, "device memory, idle stages given back");
  // What cannot be had at all is refused, and the next call served.
  expect(!HostStage::acquire(50 * MB, &e) && e == hipErrorOutOfMemory, "out of memory reported");
  (void)hipFree(p);
  big = HostStage::acquire(50 * MB, &e);
  expect(big, "a stage again");
  HostStage::release(big, true);
  HostStage::drop_idle();
  expect(g_used == 0, "everything given back");
  std::printf("host stage ok\n");
  std::fflush(stdout);
  _Exit(0);   // (helper threads sleep on)
}
