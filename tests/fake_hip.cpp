// csrc/readback.hip with the HIP runtime calls that it makes, on the host: compiled for the host alone and not linked with the
// runtime, so that its error paths and what it asks of the runtime can be tested without a GPU.
//
// Modelled is what the runtime documents and no more.  Work queued on a stream runs when somebody waits for it, or, on a stream
// that a test holds, when the test lets it go.  An event
// belongs to the device that is current when it is created and is recorded on that device's streams only.  What a kernel
// writes to pinned memory is there for the host once the kernel has run if the memory was asked for as coherent, otherwise
// behind an event that releases to the system or a stream synchronization.
#include "../turbogpt_amd/csrc/readback.hip"
#include <condition_variable>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <utility>

namespace {

struct Pinned {
    std::vector<unsigned char> host, device; // what either side sees
    unsigned flags;
    void release() { std::memcpy(host.data(), device.data(), host.size()); }
};
struct Stream {
    int device;
    std::deque<std::function<void()>> queue;
    bool held = false; // a kernel in front of the queue still runs
    bool step() {
        if (queue.empty())
            return false;
        queue.front()();
        queue.pop_front();
        return true;
    }
};
struct Event {
    int device;
    unsigned flags;
    Stream *stream;
    bool pending;
};
std::recursive_mutex guard;
std::condition_variable_any released;
int waiting = 0; // threads that wait for a held stream
typedef std::lock_guard<std::recursive_mutex> Lock;
std::map<void *, Pinned *> pinned; // by the host's address
std::map<const void *, std::string> kernels;
std::map<std::string, int> failing; // call -> fails at this call from now (1 = the next)
int events = 0;
thread_local int current_device = 0;
thread_local hipStream_t launch_stream;
thread_local hipError_t last_error = hipSuccess;

bool fails(const char *call) {
    auto at = failing.find(call);
    return at != failing.end() && at->second > 0 && --at->second == 0;
}
void release_all() {
    for (auto &entry : pinned)
        entry.second->release();
}
void run(bool join, const std::vector<uint64_t> &args) { // in, out, n or hi, lo, out, n
    unsigned char *out = reinterpret_cast<unsigned char *>(args[join ? 2 : 1]);
    const size_t bytes = args[join ? 3 : 2] * 16;
    for (auto &entry : pinned) {
        Pinned &p = *entry.second;
        if (out < p.device.data() || out + bytes > p.device.data() + p.device.size())
            continue;
        for (size_t i = 0; join && i < bytes / 4; ++i)
            reinterpret_cast<uint32_t *>(out)[i] =
                uint32_t(reinterpret_cast<uint16_t *>(args[0])[i]) << 16 | reinterpret_cast<uint16_t *>(args[1])[i];
        if (!join)
            std::memcpy(out, reinterpret_cast<void *>(args[0]), bytes);
        if (p.flags & hipHostMallocCoherent)
            p.release();
        return;
    }
    std::abort(); // a kernel writes outside the pinned memory
}

} // namespace

thread_local std::string tg_last_error;

extern "C" {

hipError_t hipGetLastError() { return std::exchange(last_error, hipSuccess); }
const char *hipGetErrorString(hipError_t error) { return error == hipErrorInvalidHandle ? "invalid handle" : "injected failure"; }
hipError_t hipSetDevice(int device) {
    current_device = device;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **out, size_t bytes, unsigned flags) {
    const Lock lock(guard);
    if (fails("hipHostMalloc"))
        return hipErrorOutOfMemory;
    Pinned *p = new Pinned{std::vector<unsigned char>(bytes, 0xee), std::vector<unsigned char>(bytes, 0xee), flags};
    pinned[p->host.data()] = p;
    *out = p->host.data();
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **out, void *host, unsigned) {
    const Lock lock(guard);
    if (fails("hipHostGetDevicePointer") || !pinned.count(host))
        return hipErrorInvalidValue;
    *out = pinned[host]->device.data();
    return hipSuccess;
}
hipError_t hipHostFree(void *host) {
    const Lock lock(guard);
    delete pinned.at(host);
    pinned.erase(host);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *out, unsigned flags) {
    const Lock lock(guard);
    if (fails("hipEventCreateWithFlags"))
        return hipErrorOutOfMemory;
    ++events;
    *out = reinterpret_cast<hipEvent_t>(new Event{current_device, flags, nullptr, false});
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t event) {
    const Lock lock(guard);
    --events;
    delete reinterpret_cast<Event *>(event);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t handle, hipStream_t stream) {
    const Lock lock(guard);
    Event *event = reinterpret_cast<Event *>(handle);
    if (fails("hipEventRecord"))
        return hipErrorUnknown;
    event->stream = reinterpret_cast<Stream *>(stream);
    if (event->device != event->stream->device)
        return hipErrorInvalidHandle;
    event->pending = true;
    event->stream->queue.push_back([event] {
        event->pending = false;
        if (event->flags & hipEventReleaseToSystem)
            release_all();
    });
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t handle) {
    std::unique_lock<std::recursive_mutex> lock(guard);
    Event *event = reinterpret_cast<Event *>(handle);
    if (fails("hipEventSynchronize"))
        return hipErrorUnknown;
    ++waiting;
    released.wait(lock, [&] { return !event->pending || !event->stream->held; });
    --waiting;
    while (event->pending)
        event->stream->step();
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t stream) {
    const Lock lock(guard);
    while (reinterpret_cast<Stream *>(stream)->step())
        ;
    release_all();
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *function, dim3, dim3, void **args, size_t, hipStream_t stream) {
    const Lock lock(guard);
    if (fails("hipLaunchKernel"))
        return last_error = hipErrorLaunchFailure;
    const bool join = kernels.at(function).find("join") != std::string::npos;
    std::vector<uint64_t> values; // they live on the launching thread's stack
    for (int i = 0; i < (join ? 4 : 3); ++i)
        values.push_back(*static_cast<uint64_t *>(args[i]));
    reinterpret_cast<Stream *>(stream)->queue.push_back([join, values] { run(join, values); });
    return hipSuccess;
}
// what the compiler's launch stubs and start-up code refer to
extern const char __hip_fatbin[] = "";
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t stream) {
    launch_stream = stream;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *shared, hipStream_t *stream) {
    *shared = 0, *stream = launch_stream;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
    kernels[host] = name;
}

// ---- for the tests -------------------------------------------------------------------------------------
void *fake_stream(int device) { return new Stream{device}; }
void fake_hold(void *stream, int held) {
    const Lock lock(guard);
    static_cast<Stream *>(stream)->held = held;
    released.notify_all();
}
int fake_waiting() {
    const Lock lock(guard);
    return waiting;
}
int fake_queued(void *stream) { return int(static_cast<Stream *>(stream)->queue.size()); }
void fake_fail(const char *call, int in) { failing[call] = in; }
int fake_pinned() { return int(pinned.size()); }
int fake_events() { return events; }

void *readback_open(int device) {
    current_device = device;
    return new std::shared_ptr<Readback>(Readback::shared(device));
}
void readback_close(void *handle) { delete static_cast<std::shared_ptr<Readback> *>(handle); }
// plain copies of `count` pieces, or joins where lo[i] is given, with every second chunk on `second` unless that is null; 0, or -1 with
// the message in readback_error()
int readback_fetch_by_two(void *handle, void *stream, void *second, int device, int count, void **host, const size_t *bytes, void **source,
                          void **lo) {
    current_device = device;
    return guarded([&] {
        std::vector<ReadbackPiece> pieces;
        for (int i = 0; i < count; ++i)
            pieces.push_back({host[i], bytes[i], lo[i] ? nullptr : source[i], static_cast<uint16_t *>(lo[i] ? source[i] : nullptr),
                              static_cast<uint16_t *>(lo[i])});
        (*static_cast<std::shared_ptr<Readback> *>(handle))->fetch(static_cast<hipStream_t>(stream), pieces, static_cast<hipStream_t>(second));
    });
}
int readback_fetch(void *handle, void *stream, int device, int count, void **host, const size_t *bytes, void **source, void **lo) {
    return readback_fetch_by_two(handle, stream, nullptr, device, count, host, bytes, source, lo);
}
const char *readback_error() { return tg_last_error.c_str(); }
}
