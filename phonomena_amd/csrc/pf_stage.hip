// Staged transfers (pf_stage.hpp): the lanes of each device and the host
// threads that work them.
#include "pf_stage.hpp"

#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>

#include "pf_runtime.hpp"

namespace pf {
namespace {

constexpr int MAX_DEVICES = 64;

struct Lane {
    hipStream_t stream = nullptr;
    char* chunk[2] = {};
    hipEvent_t done[2] = {};
};
struct Device {
    std::mutex use;              // held for a transfer
    Lane lane[STAGE_LANES];      // those made so far, from the front
    hipEvent_t ready = nullptr;
    std::mutex count;
    int users = 0;               // contexts
};
Device g_dev[MAX_DEVICES];

void destroy(Lane& l) {
    for (int k = 0; k < 2; k++) {
        if (l.chunk[k]) (void)hipHostFree(l.chunk[k]);
        if (l.done[k]) (void)hipEventDestroy(l.done[k]);
    }
    if (l.stream) (void)hipStreamDestroy(l.stream);
    l = Lane();
}

hipError_t create(Lane& l) {
    hipError_t e = hipStreamCreateWithFlags(&l.stream, hipStreamNonBlocking);
    for (int k = 0; k < 2; k++) {
        if (e == hipSuccess) e = hipHostMalloc((void**)&l.chunk[k], STAGE_CHUNK, hipHostMallocDefault);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&l.done[k], hipEventDisableTiming);
    }
    return e;
}

// Runs work(lane) on as many lanes as the transfer has chunks for, the
// caller's thread among them; lanes whose thread cannot start run here.
template <class F>
hipError_t on_lanes(int dev, size_t chunks, F work) {
    const int lanes = (int)(chunks < (size_t)STAGE_LANES ? chunks : STAGE_LANES);
    hipError_t err[STAGE_LANES];
    for (auto& e : err) e = hipSuccess;
    std::thread t[STAGE_LANES];
    for (int w = 1; w < lanes; w++) {
        try {
            t[w] = std::thread([&, w] {
                err[w] = hipSetDevice(dev);
                if (err[w] == hipSuccess) err[w] = work(w, lanes);
            });
        } catch (const std::system_error&) {
        }
    }
    err[0] = work(0, lanes);
    for (int w = 1; w < lanes; w++) {
        if (t[w].joinable()) t[w].join();
        else err[w] = work(w, lanes);
    }
    for (int w = 0; w < lanes; w++)
        if (err[w] != hipSuccess) return err[w];
    return hipSuccess;
}

// The device with the lanes that a transfer of `bytes` works, made on first
// use, for as long as `lock` is held; null when they are taken or cannot be
// made.  Device dev is current.
Device* lanes_of(int dev, size_t bytes, std::unique_lock<std::mutex>& lock) {
    if (dev < 0 || dev >= MAX_DEVICES) return nullptr;
    Device& d = g_dev[dev];
    lock = std::unique_lock<std::mutex>(d.use, std::try_to_lock);
    if (!lock.owns_lock()) return nullptr;
    hipError_t e = d.ready ? hipSuccess : hipEventCreateWithFlags(&d.ready, hipEventDisableTiming);
    for (int w = 0; w < STAGE_LANES && (size_t)w * STAGE_CHUNK < bytes && e == hipSuccess; w++)
        if (!d.lane[w].stream && (e = create(d.lane[w])) != hipSuccess) destroy(d.lane[w]);
    if (e == hipSuccess) return &d;
    (void)hipGetLastError();
    return nullptr;
}

// Frees the lanes from `first` on.
void give_back(Device& d, int first) {
    std::lock_guard<std::mutex> lock(d.use);
    for (int w = first; w < STAGE_LANES; w++) destroy(d.lane[w]);
    if (first == 0 && d.ready) {
        (void)hipEventDestroy(d.ready);
        d.ready = nullptr;
    }
}

// A copy on the device's side of PCIe: n8 eight-byte words.  A kernel moves a
// chunk as fast as the copy engine and starts sooner.
__global__ __launch_bounds__(256) void k_stage_copy(const uint2* __restrict__ src, uint2* __restrict__ dst, size_t n8) {
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < n8; t += (size_t)gridDim.x * 256) dst[t] = src[t];
}
hipError_t copy8(hipStream_t s, void* dst, const void* src, size_t bytes) {
    const size_t n8 = bytes / 8;
    const unsigned g = (unsigned)((n8 + 255) / 256 < 1024 ? (n8 + 255) / 256 : 1024);
    hipLaunchKernelGGL(k_stage_copy, dim3(g), dim3(256), 0, s, (const uint2*)src, (uint2*)dst, n8);
    return hipGetLastError();
}

}  // namespace

int stage_out(int dev, hipStream_t after, void* host, size_t bytes, const StageFill& fill, bool* taken) {
    const OnDevice on(dev);
    HIPCHK(on.error);
    std::unique_lock<std::mutex> lock;
    Device* const st = lanes_of(dev, bytes, lock);
    *taken = st != nullptr;
    if (!st || !bytes) return PF_OK;
    const size_t chunks = (bytes + STAGE_CHUNK - 1) / STAGE_CHUNK;
    if (chunks == 1) {  // nothing to overlap: in the stream's own order
        HIPCHK(fill(after, st->lane[0].chunk[0], 0, bytes));
        HIPCHK(hipStreamSynchronize(after));
        memcpy(host, st->lane[0].chunk[0], bytes);
        return PF_OK;
    }
    HIPCHK(hipEventRecord(st->ready, after));
    const hipError_t e = on_lanes(dev, chunks, [&](int w, int lanes) {
        Lane& l = st->lane[w];
        hipError_t r = hipStreamWaitEvent(l.stream, st->ready, 0);
        auto len = [&](size_t c) { return c + 1 < chunks ? STAGE_CHUNK : bytes - c * STAGE_CHUNK; };
        auto issue = [&](size_t c, int k) {
            if (r == hipSuccess) r = fill(l.stream, l.chunk[k], c * STAGE_CHUNK, len(c));
            if (r == hipSuccess) r = hipEventRecord(l.done[k], l.stream);
        };
        int k = 0;
        issue((size_t)w, 0);
        for (size_t c = (size_t)w; c < chunks && r == hipSuccess; c += (size_t)lanes, k ^= 1) {
            if (c + (size_t)lanes < chunks) issue(c + (size_t)lanes, k ^ 1);
            if (r == hipSuccess) r = hipEventSynchronize(l.done[k]);
            if (r == hipSuccess) memcpy((char*)host + c * STAGE_CHUNK, l.chunk[k], len(c));
        }
        if (r != hipSuccess) (void)hipStreamSynchronize(l.stream);  // nothing writes the chunks any more
        return r;
    });
    if (e != hipSuccess) return fail(PF_ERR_HIP, "transfer to the host: %s", hipGetErrorString(e));
    return PF_OK;
}

int stage_in(int dev, hipStream_t after, const void* host, size_t bytes, const StageDrain& drain, bool* taken) {
    const OnDevice on(dev);
    HIPCHK(on.error);
    std::unique_lock<std::mutex> lock;
    Device* const st = lanes_of(dev, bytes, lock);
    *taken = st != nullptr;
    if (!st || !bytes) return PF_OK;
    const size_t chunks = (bytes + STAGE_CHUNK - 1) / STAGE_CHUNK;
    if (chunks == 1) {
        memcpy(st->lane[0].chunk[0], host, bytes);
        HIPCHK(drain(after, st->lane[0].chunk[0], 0, bytes));
        HIPCHK(hipStreamSynchronize(after));
        return PF_OK;
    }
    HIPCHK(hipEventRecord(st->ready, after));
    const hipError_t e = on_lanes(dev, chunks, [&](int w, int lanes) {
        Lane& l = st->lane[w];
        hipError_t r = hipStreamWaitEvent(l.stream, st->ready, 0);
        int k = 0, used = 0;
        for (size_t c = (size_t)w; c < chunks && r == hipSuccess; c += (size_t)lanes, k ^= 1, used++) {
            const size_t len = c + 1 < chunks ? STAGE_CHUNK : bytes - c * STAGE_CHUNK;
            if (used >= 2) r = hipEventSynchronize(l.done[k]);
            if (r != hipSuccess) break;
            memcpy(l.chunk[k], (const char*)host + c * STAGE_CHUNK, len);
            r = drain(l.stream, l.chunk[k], c * STAGE_CHUNK, len);
            if (r == hipSuccess) r = hipEventRecord(l.done[k], l.stream);
        }
        const hipError_t s = hipStreamSynchronize(l.stream);
        return r != hipSuccess ? r : s;
    });
    if (e != hipSuccess) return fail(PF_ERR_HIP, "transfer to the device: %s", hipGetErrorString(e));
    return PF_OK;
}

int copy_out(int dev, hipStream_t after, void* host, const void* src, size_t bytes) {
    bool taken = false;
    const int rc = stage_out(dev, after, host, bytes, [=](hipStream_t s, char* dst, size_t off, size_t len) {
        return copy8(s, dst, (const char*)src + off, len);
    }, &taken);
    if (taken) return rc;
    HIPCHK(hipMemcpyAsync(host, src, bytes, hipMemcpyDeviceToHost, after));
    HIPCHK(hipStreamSynchronize(after));
    return PF_OK;
}

int copy_in(int dev, hipStream_t after, void* dst, const void* host, size_t bytes) {
    bool taken = false;
    const int rc = stage_in(dev, after, host, bytes, [=](hipStream_t s, const char* src, size_t off, size_t len) {
        return copy8(s, (char*)dst + off, src, len);
    }, &taken);
    if (taken) return rc;
    HIPCHK(hipMemcpyAsync(dst, host, bytes, hipMemcpyHostToDevice, after));
    HIPCHK(hipStreamSynchronize(after));
    return PF_OK;
}

void stage_users(int dev, int change) {
    if (dev < 0 || dev >= MAX_DEVICES) return;
    Device& d = g_dev[dev];
    bool last;
    {
        std::lock_guard<std::mutex> lock(d.count);
        d.users += change;
        last = change < 0 && d.users == 0;
    }
    if (last) give_back(d, 1);
}

}  // namespace pf

extern "C" int pf_trim(void) {
    int cur = 0;
    if (hipGetDevice(&cur) != hipSuccess) return PF_OK;  // no device, nothing kept
    for (int i = 0; i < pf::MAX_DEVICES; i++) pf::give_back(pf::g_dev[i], 0);
    return PF_OK;
}
