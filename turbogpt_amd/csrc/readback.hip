// Moves results (weights, gradients, logits, losses) into the caller's pageable memory.
//
// What bounds it is PCIe (57 GB/s measured into pinned memory) and, behind it, the host: one core copies and
// faults in fresh pages at a few GB/s.  So the result is cut into chunks; a kernel writes a chunk straight into pinned
// memory (joining the weight halves on the way, which a host loop did before), and several host threads, each with
// two buffers of its own, copy finished chunks into the caller's pages while the next ones cross the bus.  What is left
// behind the last chunk is one thread's copy of it (90 us for 2 MiB), so the last 2 MiB are cut in halves down to 512 KiB; not
// smaller, as every chunk costs its stream 6 us for its event: a large result goes by two streams in turn, so that the bus has one
// chunk while the other's event is written (a small one's first chunk would only come later).  The first chunks go out behind what is on the stream, while that still
// runs; the caller's thread alone waits for it, and the others start with the first chunk that is there (the next ones take 37 us
// each to arrive, longer than a thread takes to start): a batch's 16 MB of gradient and logits at d256 812 us with
// every thread at its own chunks from the start, 751 so.
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
void Readback::release(const Buffer &buffer) {
    if (buffer.written)
        (void)hipEventDestroy(buffer.written);
    if (buffer.pinned)
        (void)hipHostFree(buffer.pinned);
}
Readback::~Readback() {
    for (const Buffer &buffer : idle)
        release(buffer);
}
Readback::Buffer Readback::make() const { // whole or not at all
    Buffer buffer;
    try {
        check_hip(hipHostMalloc(&buffer.pinned, CHUNK, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent),
                  "pinned staging: ");
        check_hip(hipHostGetDevicePointer(&buffer.mapped, buffer.pinned, 0), "pinned staging: ");
        check_hip(hipEventCreateWithFlags(&buffer.written, hipEventDisableTiming | hipEventReleaseToSystem), "readback event: ");
    } catch (...) {
        release(buffer);
        throw;
    }
    return buffer;
}
struct Readback::Held {
    Readback &pool;
    std::vector<Buffer> buffers;
    Held(Readback &pool_, size_t count) : pool(pool_) {
        buffers.reserve(count);
        size_t missing;
        {
            const std::lock_guard<std::mutex> lock(pool.guard);
            const size_t found = std::min(count, pool.idle.size());
            missing = count - found;
            pool.idle.reserve(pool.made + missing); // giving back does not fail
            pool.made += missing;
            buffers.insert(buffers.end(), pool.idle.end() - found, pool.idle.end());
            pool.idle.resize(pool.idle.size() - found);
        }
        try {
            for (; missing; --missing)
                buffers.push_back(pool.make());
        } catch (...) {
            give_back(missing);
            throw;
        }
    }
    ~Held() { give_back(0); }
    void give_back(size_t never_made) {
        const std::lock_guard<std::mutex> lock(pool.guard);
        pool.made -= never_made;
        pool.idle.insert(pool.idle.end(), buffers.begin(), buffers.end());
    }
};

void Readback::fetch(hipStream_t stream, const std::vector<ReadbackPiece> &pieces, hipStream_t second) {
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
    if (!lanes)
        return;
    check_hip(hipSetDevice(device)); // its events are made here
    const Held held(*this, lanes * depth);
    const auto buffer = [&](size_t l, size_t round) -> const Buffer & { return held.buffers[l * depth + round % depth]; };
    const auto drain = [&] {
        (void)hipStreamSynchronize(stream);
        if (second)
            (void)hipStreamSynchronize(second);
    };
    const auto start = [&](size_t l, size_t round) {
        const size_t c = l + round * lanes;
        if (c >= chunks.size())
            return;
        const hipStream_t on = second && (c & 1) ? second : stream;
        enqueue(on, *chunks[c].piece, chunks[c].offset, chunks[c].bytes, buffer(l, round).mapped);
        check_hip(hipEventRecord(buffer(l, round).written, on));
    };
    const auto wait = [&](size_t l, size_t round) { check_hip(hipEventSynchronize(buffer(l, round).written), "readback: "); };
    const auto lane = [&](size_t l) {
        for (size_t round = 0; l + round * lanes < chunks.size(); ++round) {
            const Chunk &c = chunks[l + round * lanes];
            if (l || round) // the first chunk has been waited for
                wait(l, round);
            std::memcpy(static_cast<uint8_t *>(c.piece->host) + c.offset, buffer(l, round).pinned, c.bytes);
            start(l, round + depth);
        }
    };
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
        for (size_t round = 0; round < depth; ++round)
            for (size_t l = 0; l < lanes; ++l)
                start(l, round);
        wait(0, 0);
    } catch (...) {
        drain(); // nothing may still write to the staging buffers
        throw;
    }
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
            drain(); // as above
            std::rethrow_exception(failure);
        }
}
