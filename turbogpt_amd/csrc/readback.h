// Results to the caller's pageable host memory: see readback.hip.
#pragma once
#include "common.h"
#include <memory>
#include <mutex>
#include <vector>

// One piece of a result: `bytes` (a multiple of 16) at `host`, from a plain device buffer, or joined from the two
// 16-bit halves of fp32 values.
struct ReadbackPiece {
    void *host;
    size_t bytes;
    const void *device;               // plain copy, or
    const uint16_t *hi = nullptr, *lo = nullptr; // value i = hi[i] : lo[i]
};

class Readback {
  public:
    // The staging memory of a device is shared by its engines in this process and given back with the last of them: pinning
    // it takes longer than most results do (1.2 ms for the 16 MB of a d256 model's gradient and logits, against 1.1 ms for the
    // whole call).  Devices do not share it: an event is recorded on streams of the device that it was made on.
    static std::shared_ptr<Readback> shared(int device);
    ~Readback();
    Readback(const Readback &) = delete;
    Readback &operator=(const Readback &) = delete;
    // Copies the pieces out behind everything already on `stream`, one of the device's; returns when they are in host memory.
    // Calls on several threads run side by side, each with buffers of its own: what is on one engine's stream may take long, and
    // another engine's result does not wait for it.
    // `second`: a stream of the caller's own behind the same work, where every second chunk goes; worth it from LARGE bytes on.
    static constexpr size_t LARGE = size_t(48) << 20;
    void fetch(hipStream_t stream, const std::vector<ReadbackPiece> &pieces, hipStream_t second = nullptr);

  private:
    explicit Readback(int device_) : device(device_) {}
    struct Buffer {
        void *pinned = nullptr, *mapped = nullptr; // the same memory, by host and by device address
        hipEvent_t written = nullptr;
    };
    struct Held; // what a call has taken
    static void release(const Buffer &buffer);
    Buffer make() const;
    const int device;
    std::mutex guard;         // of the two below, never held during a wait or a copy
    std::vector<Buffer> idle; // 2 MiB each
    size_t made = 0;          // as many as the calls at one time have needed so far, at most 16 each
};
