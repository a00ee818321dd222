// host_stage.h - copies between the caller's (pageable) memory and the device through pinned memory.
//
// hipMemcpyAsync on pageable memory costs about 0.33 ms a call from 0.8 MB on, whatever it moves, and
// reads 133 MB back in 8 ms (31 ms into pages not touched before), where the link moves pinned memory at
// 57 GB/s (0.02 ms for 0.8 MB, 2.3 ms for 133 MB) and several threads fill fresh pages in 5 ms. So
// results come back through a ring of pinned chunks, from 8 MB on with threads that copy out of the ring
// while the next chunks move (a thread costs about 0.03 ms to start); one 4K image and its sums, 158 MB:
// 14 -> 5.7 ms. On the way to the device only pieces of up to one chunk go through the ring: larger
// ones move at 20-34 GB/s from pageable memory, faster than one thread fills the ring.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace crt {

class HostStage {
  public:
    struct Copy {
        void* host;        // destination
        const void* dev;   // source
        size_t bytes;
    };
    HostStage() = default;
    HostStage(const HostStage&) = delete;
    HostStage& operator=(const HostStage&) = delete;
    ~HostStage() { release(); }
    int init(int device);
    void release();
    // Device to host behind the work on `s`; the data is there on return. One caller at a time.
    hipError_t fetch(const Copy* list, int n, hipStream_t s);
    // Host to device on `s`; `src` stays as it is until the stream has come this far.
    hipError_t push(void* dst, const void* src, size_t bytes, hipStream_t s);

  private:
    static constexpr size_t kChunk = 1u << 20;
    static constexpr int kSlots = 32, kThreads = 8;
    static constexpr size_t kParallel = 8u << 20;   // bytes from which threads help
    char* pin_ = nullptr;
    hipEvent_t ev_[kSlots] = {};
    bool used_[kSlots] = {};   // ev_ marks the slot's last copy
    int next_ = 0, device_ = 0;
    hipError_t claim(int& slot);
};

}  // namespace crt
