// Staged transfers (pf_stage.hpp): the pinned memory of each device and the
// host threads that work through it.
#include "pf_stage.hpp"

#include <cstring>
#include <mutex>
#include <thread>

#include "pf_runtime.hpp"

namespace pf {
namespace {

constexpr int MAX_DEVICES = 64;

constexpr int SLOTS = 2 * STAGE_LANES;
constexpr int GROUPS = 5;  // launches that fill all slots: 1, 1, 2, 4, 8 chunks

struct Device {
    std::mutex use;  // held for a transfer
    char* pinned = nullptr;
    size_t room = 0;
    hipEvent_t done[SLOTS] = {};  // a slot's chunk has been written or read
    hipEvent_t group[GROUPS] = {};
    std::mutex count;
    int users = 0;  // contexts
};
Device g_dev[MAX_DEVICES];

void give_back(Device& d) {
    if (d.pinned) (void)hipHostFree(d.pinned);
    d.pinned = nullptr;
    d.room = 0;
}

// At least `bytes` of pinned memory, and the events.
hipError_t reserve(Device& d, size_t bytes) {
    hipError_t e = hipSuccess;
    auto make = [&](hipEvent_t& v) {
        if (!v && e == hipSuccess) e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
    };
    for (hipEvent_t& v : d.done) make(v);
    for (hipEvent_t& v : d.group) make(v);
    if (e != hipSuccess || d.room >= bytes) return e;
    give_back(d);
    e = hipHostMalloc((void**)&d.pinned, bytes, hipHostMallocDefault);
    if (e == hipSuccess) d.room = bytes;
    else d.pinned = nullptr;
    return e;
}

// A transfer's chunks: chunk c belongs to lane c % lanes, whose chunks take
// its two slots in turn.
struct Ring {
    Device* d;
    size_t bytes, chunk, chunks;
    int lanes;
    size_t len(size_t c) const { return c + 1 < chunks ? chunk : bytes - c * chunk; }
    int slot(size_t c) const { return (int)(c % (size_t)(2 * lanes)); }
    char* at(size_t c) const { return d->pinned + (size_t)slot(c) * chunk; }
    hipEvent_t done(size_t c) const { return d->done[slot(c)]; }
};

// Runs work(lane) for every lane, lane 0 on the caller's thread; lanes whose
// thread cannot start run here.
template <class F>
hipError_t on_lanes(int dev, int lanes, F work) {
    hipError_t err[STAGE_LANES];
    for (auto& e : err) e = hipSuccess;
    std::thread t[STAGE_LANES];
    for (int w = 1; w < lanes; w++) {
        try {
            t[w] = std::thread([&, w] {
                err[w] = hipSetDevice(dev);
                if (err[w] == hipSuccess) err[w] = work(w);
            });
        } catch (...) {  // no thread, or no memory for one
        }
    }
    err[0] = work(0);
    for (int w = 1; w < lanes; w++) {
        if (t[w].joinable()) t[w].join();
        else err[w] = work(w);
    }
    for (int w = 0; w < lanes; w++)
        if (err[w] != hipSuccess) return err[w];
    return hipSuccess;
}

// The ring for a transfer of `bytes` in chunks of `chunk`, for as long as
// `lock` is held; d = null when the device's is taken or cannot be made.
// Device dev is current.
Ring ring_of(int dev, size_t bytes, size_t chunk, std::unique_lock<std::mutex>& lock) {
    Ring r = {nullptr, bytes, chunk, (bytes + chunk - 1) / chunk, 1};
    if (r.chunks > 1) r.lanes = (int)(r.chunks < (size_t)STAGE_LANES ? r.chunks : STAGE_LANES);
    if (dev < 0 || dev >= MAX_DEVICES) return r;
    Device& d = g_dev[dev];
    lock = std::unique_lock<std::mutex>(d.use, std::try_to_lock);
    if (!lock.owns_lock()) return r;
    const size_t slots = r.chunks < SLOTS ? r.chunks : SLOTS;
    if (reserve(d, slots * chunk) == hipSuccess) r.d = &d;
    else (void)hipGetLastError();
    return r;
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
    // few chunks of a small transfer would leave lanes without one, more than
    // needed cost a launch and an event each
    const size_t chunk = bytes <= (16u << 20) ? 512u << 10 : bytes <= (64u << 20) ? 1u << 20 : 2u << 20;
    std::unique_lock<std::mutex> lock;
    const Ring r = ring_of(dev, bytes, chunk, lock);
    *taken = r.d != nullptr;
    if (!r.d || !bytes) return PF_OK;
    const Device& st = *r.d;
    // every slot's first chunk before the threads start, in groups that grow:
    // the first copy starts soon, and the gaps between launches stay few
    const size_t first = r.chunks < (size_t)(2 * r.lanes) ? r.chunks : (size_t)(2 * r.lanes);
    hipEvent_t ready[SLOTS];
    hipError_t e = hipSuccess;
    for (size_t c = 0, g = 0; c < first && e == hipSuccess; g++) {
        size_t n = c < 2 ? 1 : c;
        if (n > first - c) n = first - c;
        e = fill(after, r.at(c), c * chunk, (n - 1) * chunk + r.len(c + n - 1));
        if (e == hipSuccess && r.chunks > 1) e = hipEventRecord(st.group[g], after);
        while (n--) ready[c++] = st.group[g];
    }
    if (r.chunks == 1) {
        if (e == hipSuccess) e = hipStreamSynchronize(after);
        if (e == hipSuccess) memcpy(host, r.at(0), bytes);
    } else if (e == hipSuccess) {
        e = on_lanes(dev, r.lanes, [&](int w) {
            hipError_t v = hipSuccess;
            for (size_t c = (size_t)w; c < r.chunks && v == hipSuccess; c += (size_t)r.lanes) {
                v = hipEventSynchronize(c < first ? ready[c] : r.done(c));
                if (v == hipSuccess) memcpy((char*)host + c * chunk, r.at(c), r.len(c));
                const size_t next = c + (size_t)(2 * r.lanes);  // into the slot just read
                if (v == hipSuccess && next < r.chunks) v = fill(after, r.at(next), next * chunk, r.len(next));
                if (v == hipSuccess && next < r.chunks) v = hipEventRecord(r.done(next), after);
            }
            return v;
        });
    }
    if (e == hipSuccess) return PF_OK;
    (void)hipStreamSynchronize(after);  // nothing writes the chunks any more
    return fail(PF_ERR_HIP, "transfer to the host: %s", hipGetErrorString(e));
}

int stage_in(int dev, hipStream_t after, const void* host, size_t bytes, const StageDrain& drain, bool* taken) {
    const OnDevice on(dev);
    HIPCHK(on.error);
    const size_t chunk = 2u << 20;  // the host's copy of a smaller one is shorter than its launch
    std::unique_lock<std::mutex> lock;
    const Ring r = ring_of(dev, bytes, chunk, lock);
    *taken = r.d != nullptr;
    if (!r.d || !bytes) return PF_OK;
    const hipError_t e = on_lanes(dev, r.lanes, [&](int w) {
        hipError_t v = hipSuccess;
        for (size_t c = (size_t)w; c < r.chunks && v == hipSuccess; c += (size_t)r.lanes) {
            if (c >= (size_t)(2 * r.lanes)) v = hipEventSynchronize(r.done(c));  // of the slot's last chunk
            if (v != hipSuccess) break;
            memcpy(r.at(c), (const char*)host + c * chunk, r.len(c));
            v = drain(after, r.at(c), c * chunk, r.len(c));
            if (v == hipSuccess && r.chunks > 1) v = hipEventRecord(r.done(c), after);
        }
        return v;
    });
    const hipError_t s = hipStreamSynchronize(after);  // every chunk is consumed
    if (e == hipSuccess && s == hipSuccess) return PF_OK;
    return fail(PF_ERR_HIP, "transfer to the device: %s", hipGetErrorString(e != hipSuccess ? e : s));
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
    bool first, last;
    {
        std::lock_guard<std::mutex> lock(d.count);
        first = change > 0 && d.users == 0;
        d.users += change;
        last = change < 0 && d.users == 0;
    }
    if (!first && !last) return;
    std::unique_lock<std::mutex> lock(d.use, std::try_to_lock);
    if (!lock.owns_lock()) return;  // a transfer without a context runs
    if (last && d.room > STAGE_KEEP) give_back(d);
    // the first fetch or audit of the device's first context finds it made
    const OnDevice on(dev);
    if (first && on.error == hipSuccess && reserve(d, 512u << 10) != hipSuccess) (void)hipGetLastError();
}

}  // namespace pf

extern "C" int pf_trim(void) {
    int cur = 0;
    if (hipGetDevice(&cur) != hipSuccess) return PF_OK;  // no device, nothing kept
    for (pf::Device& d : pf::g_dev) {
        std::lock_guard<std::mutex> lock(d.use);
        pf::give_back(d);
    }
    return PF_OK;
}
