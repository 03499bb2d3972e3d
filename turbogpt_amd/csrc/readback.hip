// Moves results (weights, gradients, logits, losses) into the caller's pageable memory.
//
// What bounds it is PCIe (57 GB/s measured into pinned memory) and, behind it, the host: one core copies and
// faults in fresh pages at a few GB/s.  So the result is cut into chunks; a kernel writes a chunk straight into pinned
// memory (joining the weight halves on the way, which a host loop did before), and several host threads, each with
// two buffers of its own, copy finished chunks into the caller's pages while the next ones cross the bus.  What is left
// behind the last chunk is one thread's copy of it (90 us for 2 MiB), so the last 2 MiB are cut in halves down to 512 KiB; not
// smaller, as every chunk costs the bus 6 us for its event.  The threads start while what is on the stream still runs: a batch's
// 16 MB of gradient and logits at d256 875 us behind a wait for the device and in chunks of 2 MiB, 829 so.
//
// The host reads what a kernel wrote once the event behind the kernel has passed, and nothing else stands between the two.
// So both halves of that order are asked for by name, whatever the environment's default is: coherent memory, and events
// that release to the system (same rate, 49.7 GB/s a 2 MiB chunk on one stream either way).
#include "readback.h"
#include <algorithm>
#include <cstring>
#include <exception>
#include <map>
#include <thread>

namespace {

constexpr size_t CHUNK = size_t(2) << 20, SMALLEST_CHUNK = size_t(512) << 10;
constexpr int LANES = 8;

__global__ __launch_bounds__(256) void readback_copy_kernel(const u32x4 *__restrict__ in, u32x4 *__restrict__ out,
                                                            size_t n) {
    for (size_t i = size_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += size_t(gridDim.x) * 256)
        __builtin_nontemporal_store(in[i], out + i);
}
__global__ __launch_bounds__(256) void readback_join_kernel(const u32x2 *__restrict__ hi, const u32x2 *__restrict__ lo,
                                                            u32x4 *__restrict__ out, size_t n) {
    for (size_t i = size_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += size_t(gridDim.x) * 256) {
        const u32x2 h = hi[i], l = lo[i];
        const u32x4 joined = {(h.x << 16) | (l.x & 0xffffu), (h.x & 0xffff0000u) | (l.x >> 16),
                              (h.y << 16) | (l.y & 0xffffu), (h.y & 0xffff0000u) | (l.y >> 16)};
        __builtin_nontemporal_store(joined, out + i);
    }
}

void enqueue(hipStream_t stream, const ReadbackPiece &piece, size_t offset, size_t bytes, void *out) {
    const size_t n = bytes / 16;
    const dim3 grid(unsigned(std::min<size_t>((n + 255) / 256, 512)));
    if (piece.hi)
        hipLaunchKernelGGL(readback_join_kernel, grid, dim3(256), 0, stream,
                           reinterpret_cast<const u32x2 *>(piece.hi + offset / 4),
                           reinterpret_cast<const u32x2 *>(piece.lo + offset / 4), static_cast<u32x4 *>(out), n);
    else
        hipLaunchKernelGGL(readback_copy_kernel, grid, dim3(256), 0, stream,
                           reinterpret_cast<const u32x4 *>(static_cast<const uint8_t *>(piece.device) + offset),
                           static_cast<u32x4 *>(out), n);
    check_hip(hipGetLastError(), "readback launch: ");
}

} // namespace

std::shared_ptr<Readback> Readback::shared(int device) {
    static std::mutex guard;
    static std::map<int, std::weak_ptr<Readback>> living;
    const std::lock_guard<std::mutex> lock(guard);
    std::weak_ptr<Readback> &place = living[device];
    std::shared_ptr<Readback> staging = place.lock();
    if (!staging)
        place = staging = std::shared_ptr<Readback>(new Readback(device));
    return staging;
}
void Readback::give_back(const Buffer &buffer) {
    if (buffer.written)
        (void)hipEventDestroy(buffer.written);
    if (buffer.pinned)
        (void)hipHostFree(buffer.pinned);
}
Readback::~Readback() {
    for (const Buffer &buffer : buffers)
        give_back(buffer);
}
void Readback::reserve(size_t count) {
    buffers.reserve(count);
    while (buffers.size() < count) { // a buffer joins the others whole or not at all
        Buffer buffer;
        try {
            check_hip(hipHostMalloc(&buffer.pinned, CHUNK, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent),
                      "pinned staging: ");
            check_hip(hipHostGetDevicePointer(&buffer.mapped, buffer.pinned, 0), "pinned staging: ");
            check_hip(hipEventCreateWithFlags(&buffer.written, hipEventDisableTiming | hipEventReleaseToSystem), "readback event: ");
        } catch (...) {
            give_back(buffer);
            throw;
        }
        buffers.push_back(buffer);
    }
}

void Readback::fetch(hipStream_t stream, const std::vector<ReadbackPiece> &pieces) {
    struct Chunk {
        const ReadbackPiece *piece;
        size_t offset, bytes;
    };
    std::vector<Chunk> chunks;
    size_t left = 0;
    for (const ReadbackPiece &piece : pieces) {
        require(piece.bytes % 16 == 0, "readback: size must be a multiple of 16");
        left += piece.bytes;
    }
    for (const ReadbackPiece &piece : pieces)
        for (size_t at = 0; at < piece.bytes;) {
            const size_t half = left / 2 & ~size_t(0xffff); // whole 64 KiB
            const size_t bytes = std::min(std::clamp(half, SMALLEST_CHUNK, CHUNK), piece.bytes - at);
            chunks.push_back({&piece, at, bytes});
            at += bytes, left -= bytes;
        }
    // lane `l` of `lanes` takes chunks l, l + lanes, ... with two buffers of its own in turn
    const size_t lanes = std::min<size_t>(LANES, (chunks.size() + 1) / 2);
    const size_t depth = chunks.size() == 1 ? 1 : 2;
    const std::lock_guard<std::mutex> lock(busy);
    check_hip(hipSetDevice(device)); // its events are made here
    reserve(lanes * depth);
    const auto lane = [&](size_t l) {
        const auto start = [&](size_t round) {
            const size_t c = l + round * lanes;
            if (c >= chunks.size())
                return;
            Buffer &buffer = buffers[l * depth + round % depth];
            enqueue(stream, *chunks[c].piece, chunks[c].offset, chunks[c].bytes, buffer.mapped);
            check_hip(hipEventRecord(buffer.written, stream));
        };
        for (size_t round = 0; round + 1 < depth; ++round)
            start(round);
        for (size_t round = 0; l + round * lanes < chunks.size(); ++round) {
            start(round + depth - 1);
            const Chunk &c = chunks[l + round * lanes];
            const Buffer &buffer = buffers[l * depth + round % depth];
            check_hip(hipEventSynchronize(buffer.written), "readback: ");
            std::memcpy(static_cast<uint8_t *>(c.piece->host) + c.offset, buffer.pinned, c.bytes);
        }
    };
    if (!lanes)
        return;
    std::vector<std::exception_ptr> failures(lanes);
    std::vector<std::thread> threads;
    const auto guarded_lane = [&](size_t l) {
        try {
            check_hip(hipSetDevice(device));
            lane(l);
        } catch (...) {
            failures[l] = std::current_exception();
        }
    };
    try {
        for (size_t l = 1; l < lanes; ++l)
            threads.emplace_back(guarded_lane, l);
    } catch (...) { // no more threads: this one takes the lanes that are left
        for (size_t l = threads.size() + 1; l < lanes; ++l)
            guarded_lane(l);
    }
    guarded_lane(0); // this thread; a small result has no other
    for (std::thread &thread : threads)
        thread.join();
    for (const std::exception_ptr &failure : failures)
        if (failure) {
            (void)hipStreamSynchronize(stream); // nothing may still write to the staging buffers
            std::rethrow_exception(failure);
        }
}
