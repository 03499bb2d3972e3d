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
    // whole call).  Calls on several threads take turns; they share one bus.  Devices do not share it: an event is recorded
    // on streams of the device that it was made on.
    static std::shared_ptr<Readback> shared(int device);
    ~Readback();
    Readback(const Readback &) = delete;
    Readback &operator=(const Readback &) = delete;
    // Copies the pieces out behind everything already on `stream`, one of the device's; returns when they are in host memory.
    void fetch(hipStream_t stream, const std::vector<ReadbackPiece> &pieces);

  private:
    explicit Readback(int device_) : device(device_) {}
    struct Buffer {
        void *pinned = nullptr, *mapped = nullptr; // the same memory, by host and by device address
        hipEvent_t written = nullptr;
    };
    static void give_back(const Buffer &buffer);
    void reserve(size_t count);
    const int device;
    std::mutex busy;
    std::vector<Buffer> buffers; // 2 MiB each, as many as the largest result so far could use: at most 16
};
