// Host-side context of libphonofdtd, shared by the API translation units.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/phonofdtd.h"
#include "pf_kernels.hpp"

// Flags of the events the library times launches with: no system-scope
// fence when an event is recorded (a recorded event would otherwise write
// back and invalidate the caches between the launches it brackets, which
// slows the launches after it; the elapsed times are read only after a
// stream synchronization, which makes the event visible).
#define PF_TIMING_EVENT hipEventDisableSystemFence

// Material rows the tiled sweep stages in LDS.
#define PF_TILED_MAX_MATERIALS 16
// Snapshot slots a context can hold.
#define PF_SNAP_MAX_SLOTS 16
// Offset of time level l in its allocation: l * PF_LEVEL_STAGGER bytes (an
// odd multiple of 256).
#define PF_LEVEL_STAGGER 4352
// Launch groups of each kind (pairs, single steps) that one pf_profile call
// brackets with events at most.
#define PF_PROFILE_BRACKETS 8
#define PF_PROFILE_EVENTS (4 * PF_PROFILE_BRACKETS + 1)

namespace pf {
// A partition of the mesh into ntx x nty x ntz owned boxes (balanced; at
// least 3 nodes an axis, so a box that holds a face holds the cells its Mur
// map reads) for launches of `steps` whole steps, and the threads that the
// largest box with its halo needs (pf_block.hpp).
struct BlockMap {
    int ntx, nty, ntz, steps, threads;
};
constexpr int BLOCK_MAX_STEPS = 4;
// Blocks of an energy audit: `per` a chunk of xchunk planes (pf_energy.hpp).
struct EnergyGrid {
    long long per, blocks;
    int xchunk;
};
}  // namespace pf

// One mesh on one device.  Time levels of the displacement components are
// kept in level buffers: `cur` indexes the current level (n) and `old` the
// previous one (n-1); a single step overwrites `old` with level n+1 and
// swaps the two.  Two-step sweeps and block steps use two more level
// buffers.  Each level is one allocation holding its arrays back to back
// (ux, uy, uz, then the 16-bit lo parts in FP32C), so one buffer descriptor
// covers a whole level; level l starts l * PF_LEVEL_STAGGER bytes into its
// allocation (lvlbase[l] is the allocation, lvl[l][0] the level).
struct pf_ctx {
    int nx = 0, ny = 0, nz = 0, pz = 0;
    long long plane = 0, cells = 0;  // ny*pz, nx*ny*pz
    int precision = 0, kernel = 0, tile_j = 4, tile_x = 0, tile_z = 64;
    int pair_j = 0, pair_z = 0;  // tile of the two-step sweep (PF_KERNEL_TILED2)
    bool shape_open = false;     // tile shape left to measurement at creation
    // planes per x chunk of the one-step sweep, for the shape and resident
    // blocks it was last chosen for (tile_map)
    mutable struct {
        int tj = 0, kz = 0;
        long long slots = 0;
        int xchunk = 0;
    } auto_chunk;
    // a small mesh: whole steps in blocks, block_steps a launch at most, with
    // the partition for r steps at block[r]
    int block_steps = 0;
    pf::BlockMap block[pf::BLOCK_MAX_STEPS + 1] = {};
    size_t esz = 8;
    bool sponge = false;
    int surface = 0;  // pf_desc.surface
    double dt = 0;
    int nmat = 0;
    int dev = 0;
    int cus = 0;  // compute units of the device (0: unknown)
    hipStream_t stream = nullptr;
    void* lvlbase[4] = {};
    void* lvl[4][3] = {};
    void* lvlo[4][3] = {};
    int nlevels = 0;
    int cur = 0, old = 1;
    uint8_t* ids = nullptr;
    void *mat = nullptr, *fx = nullptr, *fy = nullptr, *fz = nullptr, *sx = nullptr, *sy = nullptr,
         *sz = nullptr;
    void *dpx = nullptr, *dpy = nullptr, *dpz = nullptr;
    // FP64: the reciprocals of the spacing tables, which fx.. keep.  recip:
    // every spacing is a power of two, so the tiled sweep and block steps
    // multiply by them (MODE_FP64P); quot: otherwise the tiled sweep takes exact
    // quotients from them (MODE_FP64Q); quot_open: it might, the spacings are
    // not tried (take_quotients).
    bool recip = false, quot = false, quot_open = false;
    void *rfx = nullptr, *rfy = nullptr, *rfz = nullptr, *rsx = nullptr, *rsy = nullptr, *rsz = nullptr;
    void *mat64 = nullptr, *rho64 = nullptr, *fx64 = nullptr, *fy64 = nullptr, *fz64 = nullptr,
         *sx64 = nullptr, *sy64 = nullptr, *sz64 = nullptr;
    double f0[3] = {}, s0[3] = {};
    double dV = 0;
    double mur[12] = {};
    double* wave = nullptr;
    long long wave_len = 0;
    long long* d_step = nullptr;  // device step counter (graph replays)
    long long step = 0;           // steps issued
    int probe[6] = {};
    int every = 0, cap = 0;
    double* ring = nullptr;
    long long* d_frame = nullptr;  // [0] frames recorded; [1], as an int: blocks done in the probe launch
    // energy audit: the blocks' partial sums, then room for the two sums
    pf::EnergyGrid e_grid = {};
    double* e_partials = nullptr;
    void* scratch = nullptr;
    size_t scratch_bytes = 0;
    pf_batch* batch = nullptr;  // set while a batch owns the stepping
    hipStream_t batch_stream = nullptr;
    // asynchronous snapshots: per slot a device staging frame and a pinned
    // host frame (ux, uy, uz in the reference's shapes, FP64), the copy on
    // its own stream
    int snap_slots = 0;
    long long snap_frame = 0;  // doubles per frame
    double* snap_dev = nullptr;
    double* snap_host = nullptr;
    hipStream_t snap_stream = nullptr;
    hipEvent_t snap_packed[PF_SNAP_MAX_SLOTS] = {};
    hipEvent_t snap_copied[PF_SNAP_MAX_SLOTS] = {};
    int snap_state[PF_SNAP_MAX_SLOTS] = {};      // 0 free, 1 in flight, 2 held by the caller
    long long snap_step[PF_SNAP_MAX_SLOTS] = {};
    // pf_profile's timing events, created by its first call and kept, so
    // that later calls time the steps and not the event set-up
    hipEvent_t prof_ev[PF_PROFILE_EVENTS] = {};
};

namespace pf {

// Bytes of one time level: three components of esz bytes, plus three
// 16-bit lo parts in PF_FP32C.
inline unsigned long long level_bytes(long long cells, int precision) {
    const unsigned long long c = (unsigned long long)cells;
    if (precision == PF_FP64) return c * 3 * 8;
    return c * 3 * 4 + (precision == PF_FP32C ? c * 3 * sizeof(lo_t) : 0);
}

int fail(int code, const char* fmt, ...);

// Device dev current for a scope: a caller may have another one current when
// it uses a context, and what is made for the context (memory, streams,
// events) has to be on the context's device.
struct OnDevice {
    hipError_t error;
    int was = -1;
    explicit OnDevice(int dev) {
        int cur = -1;
        error = hipGetDevice(&cur);
        if (error != hipSuccess || cur == dev) return;
        error = hipSetDevice(dev);
        if (error == hipSuccess) was = cur;
    }
    ~OnDevice() {
        if (was >= 0) (void)hipSetDevice(was);
    }
    OnDevice(const OnDevice&) = delete;
    OnDevice& operator=(const OnDevice&) = delete;
};

int ctx_init(pf_ctx* c, const pf_desc* d);
void ctx_free(pf_ctx* c);
void take_quotients(pf_ctx* c);
// View of a step from level `cur` (n) and `old` (n-1) into level `out`.
template <class R>
Mesh<R> make_view(const pf_ctx* c, int cur, int old, int out);
// Issue one step (sweep, faces, probe) on stream s; tt = *base + off (or
// off when base is null).  ev: 2 events recorded before and after the
// sweep, or null.
int step_once(pf_ctx* c, hipStream_t s, const long long* base, long long off, hipEvent_t* ev);
// Issue steps tt and tt+1 with the two-step sweep (PF_KERNEL_TILED2); ev as
// for step_once (around the two-step pass).
int step_pair(pf_ctx* c, hipStream_t s, const long long* base, long long off, hipEvent_t* ev);
// Device address of the allocation-free staging array on device dev, taken
// once per device (called at context creation, with dev current).
int noalloc_scratch_init(int dev);

}  // namespace pf

#define HIPCHK(x)                                                                                   \
    do {                                                                                            \
        hipError_t e_ = (x);                                                                        \
        if (e_ != hipSuccess)                                                                       \
            return pf::fail(PF_ERR_HIP, "%s failed: %s (%s:%d)", #x, hipGetErrorString(e_), __FILE__, \
                            __LINE__);                                                              \
    } while (0)
