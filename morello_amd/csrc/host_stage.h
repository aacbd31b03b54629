// Device and pinned memory for Specs called on host buffers (mrl_run_host), kept between calls.
//
// A parameter on the host reaches the GPU through pinned memory: the caller and, for transfers of
// megabytes, a few helper threads copy it there piece by piece, and a copy kernel takes each piece
// across PCIe behind them; results come back the same way, a flag in pinned memory telling the host
// when a piece has landed.  Measured on this part (GB/s of PCIe Gen5 x16, 57 at most): pageable
// hipMemcpy 31-37 in and 17 out from 4 MiB on but 2-3 at 128 KiB to 1 MiB, one host thread's
// memcpy 31, two 57, four 84; the copy kernel on 16 workgroups 55.  A tiny launch and
// hipStreamSynchronize take 11 us, a launch whose flag the host polls about 8.  In and out again through
// a Move (us, hipMalloc + hipMemcpy + hipFree per call / this): 4 KiB 50 / 17, 128 KiB 48 / 27, 1 MiB 126 /
// 89, 8 MiB 841 / 447, 64 MiB 6655 / 2851 (47 GB/s each way).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>

namespace mrl {

class HostStage {
 public:
  // A stage of the current device that no other thread uses, with `bytes` of device memory; nullptr
  // and *err on failure.  Give it back with release().
  static HostStage *acquire(size_t bytes, hipError_t *err);
  // Idle stages stay for later calls (at most IDLE_MAX of them, each with at most KEEP_DEVICE_BYTES)
  // once their work is complete; a stage whose call failed (`good` false) does not.
  static void release(HostStage *stage, bool good);
  // Frees the idle stages and the scratch kept for their streams; whether there were any.
  static bool drop_idle();
  static constexpr int IDLE_MAX = 2;

  struct Piece {      // a parameter: `bytes` at `offset` (a multiple of 256) of the device memory
    void *host;
    size_t offset, bytes;
  };
  // Enqueues host -> device copies of the pieces on the stage's stream; the host memory has been read
  // when it returns.
  hipError_t upload(const Piece *pieces, int n);
  // Enqueues device -> host copies behind the work on the stage's stream and waits for all of it.
  hipError_t download(const Piece *pieces, int n);

  uint8_t *device() const { return dev_; }
  hipStream_t stream() const { return stream_; }

 private:
  static constexpr size_t KEEP_DEVICE_BYTES = size_t(1) << 30, PINNED_BYTES = size_t(32) << 20;
  static constexpr size_t PART_MAX = size_t(2) << 20;   // what one copy kernel takes at most: 37 us of PCIe against a launch's ~2
  static constexpr int SLOTS = int(PINNED_BYTES / PART_MAX);
  struct Parts;
  HostStage() = default;
  ~HostStage();
  hipError_t init();
  hipError_t wait(uint32_t slot, uint32_t ticket, const std::atomic<int> &failed);
  hipError_t copy(void *dst, const void *src, size_t bytes, uint32_t slot, uint32_t ticket, hipStream_t stream);

  int device_id_ = 0;
  hipStream_t stream_ = nullptr, side_ = nullptr;   // the Spec's and half of the copies; the other half
  hipEvent_t join_ = nullptr;
  uint8_t *dev_ = nullptr, *pin_ = nullptr;
  size_t dev_size_ = 0;
  uint32_t *flags_ = nullptr;     // pinned: the ticket of the last copy that is complete, per slot
  uint32_t *counters_ = nullptr;  // device: workgroups of a copy that are done, per slot
  uint32_t ticket_ = 0;
};

// hipMalloc for all of the library's device memory: where there is not enough, what idle stages keep is given back
// and tried for once more.
hipError_t device_malloc(void **p, size_t bytes);

// What to call with a stage's stream before it is destroyed (the scratch arena kept for it).
void on_host_stage_stream_end(void (*f)(hipStream_t));

}  // namespace mrl
