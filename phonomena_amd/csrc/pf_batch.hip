// Batched stepping: many contexts of one precision stepped together.
//
// Per step the batch issues two launches whatever its size:
//   1. one persistent sweep over a combined tile work-list of all members
//      (the same per-tile code as the single-mesh tiled sweep, so a member's
//      fields are bit-identical to stepping it alone);
//   2. one launch over all members' boundary-face cells, which records their
//      probe frames too.
// The steps since the tables were built are counted on the device (a launch
// takes its place in a group of steps as an argument, and one small launch
// per group moves the counters on), and which of a member's two levels is
// current follows from that, so K steps are captured once in a HIP graph and
// replayed.  A member whose step index reaches its source-table length (its
// step budget) stops: its tiles, faces and probes return at once and its
// counters no longer move.
//
// Work-list: the tiles of every member, member after member in tile order,
// cut into 8 contiguous runs of equal plane count, one per XCD (the device
// hands out workgroups to XCDs round-robin, so block b runs on XCD b % 8).
// Each block takes the next tile of its XCD's run from an atomic counter,
// so neighbouring tiles, which share halo rows, are swept on the same L2.
// The counters of a step are reset by the previous step's launch.
//
// Tile shapes (rows x lanes and planes per chunk) are the batch's; the
// autotuner times candidate shapes on real steps (every shape gives the
// same bits) and keeps the fastest.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstring>
#include <vector>

#include "pf_runtime.hpp"
#include "pf_tiled.hpp"

using namespace pf;

namespace pf {

constexpr int NXCD = 8;

template <class R>
struct BMember {
    Mesh<R> view[2];        // mesh views with level 0 / level 1 current
    TileMap tm;
    long long* step;        // the member's device step counter
    long long t0;           // its step count when the views were taken (view[0])
    FaceProbe probe;        // ni = 0: none
    int row_blocks, edge_blocks;  // as face_rows_grid gives them
    long long budget;       // source-table length
};

// The member table is read through the constant address space: its loads
// are scalar (one per block, into scalar registers), as a kernel argument's
// are.  Through a plain pointer every use of a mesh field inside the march
// became a vector load with a full wait.
template <class R>
using CMember = const __attribute__((address_space(4))) BMember<R>;

struct WorkItem {
    int member, tile;
};
typedef const __attribute__((address_space(4))) WorkItem CItem;

// A copy of *p read word by word through the constant address space
// (block-uniform p), i.e. with scalar loads.
template <class T>
PF_DEV T load_const(const T* p) {
    static_assert(sizeof(T) % 4 == 0, "word-sized struct");
    typedef const __attribute__((address_space(4))) unsigned int CWord;
    const CWord* w = (const CWord*)p;
    T v;
    unsigned int* d = (unsigned int*)&v;
#pragma unroll
    for (unsigned k = 0; k < sizeof(T) / 4; k++) d[k] = w[k];
    return v;
}

// Pointers read from memory lead to global memory, as the compiler knows of a
// kernel's arguments; otherwise it accesses them with flat instructions, which
// wait for the LDS too.
template <class... P>
PF_DEV void in_global(P&... p) {
    ((p = (P)(__attribute__((address_space(1))) std::remove_reference_t<decltype(*p)>*)(uintptr_t)p), ...);
}

// Mesh view of member i, n steps after the tables were built.
template <class R>
PF_DEV Mesh<R> current_view(const BMember<R>* mem, int i, long long n) {
    CMember<R>* cm = (CMember<R>*)mem;
    Mesh<R> m = load_const(&mem[i].view[n & 1]);
    m.step_base = nullptr;
    m.step_off = cm[i].t0 + n;
    in_global(m.c0, m.c1, m.c2, m.cl0, m.cl1, m.cl2, m.n0, m.n1, m.n2, m.nl0, m.nl1, m.nl2, m.wave, m.mat, m.sx, m.fx,
              m.sy, m.fy, m.sz, m.fz, m.rsx, m.rfx, m.rsy, m.rfy, m.rsz, m.rfz, m.dpx, m.dpy, m.dpz);
    return m;
}

template <class R, int MODE, bool SPONGE, int TJ, int KZ>
__global__ __launch_bounds__(TJ * KZ, (MODE == MODE_FP32 ? 4 : MODE == MODE_FP64Q ? 3 : 2)) void k_batch_sweep(
    const BMember<R>* __restrict__ mem, const WorkItem* __restrict__ items, const int* __restrict__ qbeg,
    int* __restrict__ ctr, const long long* __restrict__ bstep, int off) {
    __shared__ TiledLds<R, TJ, KZ, Spacing<R, MODE>> L;
    __shared__ int s_item;
    const int tid = threadIdx.y * 64 + threadIdx.x;
    const int x = (int)(blockIdx.x % NXCD);
    const long long n = *bstep + off;
    const int par = (int)(n & 1);
    if (blockIdx.x == 0 && tid < NXCD) ctr[(par ^ 1) * NXCD + tid] = 0;  // next step's counters
    int* c = ctr + par * NXCD + x;
    const int end = qbeg[x + 1];
    for (;;) {
        __syncthreads();  // the previous tile's LDS reads and s_item are done
        if (tid == 0) s_item = qbeg[x] + atomicAdd(c, 1);
        __syncthreads();
        const int it = __builtin_amdgcn_readfirstlane(s_item);
        if (it >= end) break;  // uniform: every wave of the block leaves
        CItem* ci = (CItem*)items;
        const int mi = ci[it].member, tile = ci[it].tile;
        CMember<R>* cm = (CMember<R>*)mem;
        const TileMap tm = {cm[mi].tm.nkt, cm[mi].tm.njt, cm[mi].tm.nxc, cm[mi].tm.xchunk};
        const Mesh<R> m = current_view(mem, mi, n);
        tiled_tile<R, MODE, SPONGE, TJ, KZ>(m, tm, tile, L);
    }
}

// Face block g of a batched step: its member and its index among that
// member's blocks (one table load instead of a search).
struct FaceBlock {
    int member, block;
};

// Blocks of member c's face cells and probe points.
template <class R>
int face_blocks(BMember<R>& e, const pf_ctx* c) {
    const int* q = c->probe;
    e.probe = {c->ring, c->d_frame, nullptr, q[0], q[1], q[2], q[3], q[4], q[5], c->cap, c->every,
               q[2] > 0 ? (q[2] * q[5] + 255) / 256 : 0};
    long long rb, eb;
    face_rows_grid(c->nx, c->ny, c->nz, rb, eb);
    e.row_blocks = (int)rb;
    e.edge_blocks = (int)eb;
    return (int)(rb + eb) + e.probe.blocks;
}

// Face cells and probe frames of all members: every block does what a block
// of k_faces_rows does for one mesh.  It is bound by its fixed cost and the
// chain of loads each wave makes (member, view, cells): 14.7 us at 16 members
// of 14.2 M nodes in FP32C, against 24.7 us with 1024 cells of a flat list per
// block and 6.0 us for the frames and the counters in a launch of their own;
// a step of 5 members of 1.4 M nodes went from 64 to 49 us.
template <class R, int MODE>
__global__ __launch_bounds__(256) void k_batch_faces(const BMember<R>* __restrict__ mem,
                                                     const FaceBlock* __restrict__ fmap,
                                                     const long long* __restrict__ bstep, int off) {
    const long long n = *bstep + off;
    const FaceBlock fb = load_const(&fmap[blockIdx.x]);
    CMember<R>& e = ((CMember<R>*)mem)[fb.member];
    const auto& v = e.view[n & 1];
    const long long tt = e.t0 + n;
    if (tt >= v.nsteps) return;
    const R w = (R)v.wave[tt];
    const int rows = e.row_blocks, edges = e.edge_blocks;
    // each branch takes the view by itself: what it does not use is then not
    // loaded (one view for all was 250 scalar registers more than there are)
    auto view = [&]() { return current_view(mem, fb.member, n); };
    if (fb.block < rows) {
        face_rows_block<R, MODE>(v.nx, v.ny, v.nz, view, fb.block, w);
        return;
    }
    if (fb.block < rows + edges) {
        face_edges_block<R, MODE>(view(), fb.block - rows, w);
        return;
    }
    const FaceProbe pr = load_const(&mem[fb.member].probe);
    if ((tt + 1) % pr.every != 0) return;
    const int p = (fb.block - rows - edges) * 256 + (int)threadIdx.x, np = pr.ni * pr.nj;
    if (p < np) pr.ring[(tt / pr.every) % pr.cap * np + p] = probe_point<R, MODE>(view(), pr, p, w);
}

// The counters after a group of `by` steps.  A member's frames are those its
// steps have recorded.
template <class R>
__global__ __launch_bounds__(256) void k_batch_advance(const BMember<R>* __restrict__ mem, int nmem,
                                                       long long* __restrict__ bstep, int by) {
    CMember<R>* cm = (CMember<R>*)mem;
    for (int i = threadIdx.x; i < nmem; i += 256) {
        const long long v = *cm[i].step + by, cap = cm[i].budget;
        const long long t = v < cap ? v : cap;
        *cm[i].step = t;
        if (cm[i].probe.blocks > 0) *cm[i].probe.frame = t / cm[i].probe.every;
    }
    if (threadIdx.x == 0) *bstep += by;
}

}  // namespace pf

struct pf_batch {
    int precision = 0;
    int sponge = -1;  // set by the first member
    int mode = 0;     // the sweep's, set with the tables
    std::vector<pf_ctx*> members;
    hipStream_t stream = nullptr;
    int dev = 0, cus = 0;
    int tile_j = 0, tile_z = 0, tile_x = 0;
    bool use_graph = true;
    // device tables
    void* d_mem = nullptr;
    size_t mem_bytes = 0;
    WorkItem* d_items = nullptr;
    size_t items_cap = 0;
    int* d_qbeg = nullptr;
    int* d_ctr = nullptr;
    long long* d_bstep = nullptr;
    FaceBlock* d_fmap = nullptr;
    size_t fmap_cap = 0;
    long long face_blocks = 0;
    int grid = 0;
    bool dirty = true;
    // captured step loop
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    int graph_steps = 0;
};

namespace {

int free_graph(pf_batch* b) {
    if (b->exec) HIPCHK(hipGraphExecDestroy(b->exec));
    if (b->graph) HIPCHK(hipGraphDestroy(b->graph));
    b->exec = nullptr;
    b->graph = nullptr;
    b->graph_steps = 0;
    return PF_OK;
}

void free_tables(pf_batch* b) {
    auto F = [](void* p) { if (p) (void)hipFree(p); };
    F(b->d_mem); F(b->d_items); F(b->d_qbeg); F(b->d_ctr); F(b->d_bstep); F(b->d_fmap);
    b->d_mem = nullptr; b->d_items = nullptr; b->d_qbeg = nullptr; b->d_ctr = nullptr; b->d_bstep = nullptr;
    b->d_fmap = nullptr;
    b->mem_bytes = b->items_cap = b->fmap_cap = 0;
}

// Default rows x lanes of a batch (the autotuner refines them): 16 x 32, 8 x
// 32 in FP64.  Members are a few times 30 nodes deep, so 62-lane tiles leave
// lanes idle, and 32 rows make few work items of a small batch.  Measured,
// microseconds a step at each shape's best chunk (with the earlier face and
// probe launches, 10 to 16 us more), 16 x 32 / 16 x 64 / 8 x 64 /
// 32 x 32 / 8 x 32: 16 members of 14.2 M nodes FP32C 312 / 315 / 312 / 315 /
// 335; 10 of 2.8 M 88 / 92 / 95 / 91 / 92; 5 of 1.4 M 64 / 61 / 67 / 62 / 67.
// From 2^25 nodes on, where every shape keeps the chip full, 16 x 64 (FP32 and
// FP32C), which reads fewer halo lines: 64 members of 56.6 M nodes FP32 635 us
// against 651, FP32C 1087 against 1098.  A caller that gives one of the two gets the other as it always was: 64
// lanes (32 in FP64), 16 rows of 64 or 32 of 32 (8 in FP64).
void resolve_shape(int precision, long long nodes, int& tj, int& tz) {
    const bool f64 = precision == PF_FP64;
    if (tj == 0 && tz == 0) {
        tj = f64 ? 8 : 16;
        tz = f64 || nodes < (1ll << 25) ? 32 : 64;
    }
    if (tz == 0) tz = f64 ? 32 : 64;
    if (tj == 0) tj = f64 ? 8 : (tz == 64 ? 16 : 32);
}

void batch_shape(const pf_batch* b, int& tj, int& tz) {
    tj = b->tile_j;
    tz = b->tile_z;
    long long nodes = 0;
    for (const pf_ctx* c : b->members) nodes += c->cells;
    resolve_shape(b->precision, nodes, tj, tz);
}

// Default planes per chunk: about 1.5 work items per resident block, so that
// the queues even out uneven members and no CU runs two chunks while another
// runs none, within 8 (shorter chunks repeat too many warm-up planes) and 32
// (longer ones gain nothing).  Measured at 8 / 12 / 16 / 24 / 32 / 48 planes,
// 16 x 32 FP32C: 5 members of 1.4 M nodes 65 / 64 / 70 / 84 / 91 / 108 us a
// step (the rule: 8), 10 of 2.8 M 89 / 88 / 91 / 93 / 119 / 127 (17), 16 of
// 14.2 M 330 / 318 / 314 / 312 / 312 / 328 (32).
int default_xchunk(const pf_batch* b, int tj, int tz) {
    double planes = 0;  // tile planes of all members
    for (const pf_ctx* c : b->members) {
        const TileMap tm = tile_map(c, tj, tz, 1);
        planes += (double)tm.nkt * tm.njt * c->nx;
    }
    const int tx = (int)(planes / (1.5 * b->grid) + 0.5);
    return tx < 8 ? 8 : tx > 32 ? 32 : tx;
}

bool shape_built(int tj, int tz) {
    return (tz == 64 && (tj == 8 || tj == 16)) || (tz == 32 && (tj == 8 || tj == 16 || tj == 32));
}

template <class R, int MODE, bool SPONGE, int TJ, int KZ>
int sweep_grid(pf_batch* b) {
    int per = 0;
    HIPCHK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void*)k_batch_sweep<R, MODE, SPONGE, TJ, KZ>,
                                                        TJ * KZ, 0));
    if (per < 1) per = 1;
    b->grid = per * b->cus;
    b->grid = (b->grid + NXCD - 1) / NXCD * NXCD;
    return PF_OK;
}

template <class R, int MODE, bool SPONGE>
int sweep_grid_s(pf_batch* b, int tj, int tz) {
    if (tz == 64 && tj == 16) return sweep_grid<R, MODE, SPONGE, 16, 64>(b);
    if (tz == 64 && tj == 8) return sweep_grid<R, MODE, SPONGE, 8, 64>(b);
    if (tz == 32 && tj == 32) return sweep_grid<R, MODE, SPONGE, 32, 32>(b);
    if (tz == 32 && tj == 16) return sweep_grid<R, MODE, SPONGE, 16, 32>(b);
    return sweep_grid<R, MODE, SPONGE, 8, 32>(b);
}

template <class R, int MODE>
int sweep_grid_t(pf_batch* b, int tj, int tz) {
    return b->sponge == 1 ? sweep_grid_s<R, MODE, true>(b, tj, tz) : sweep_grid_s<R, MODE, false>(b, tj, tz);
}

template <class R, int MODE>
int build_t(pf_batch* b) {
    int tj, tz;
    batch_shape(b, tj, tz);
    int rc = sweep_grid_t<R, MODE>(b, tj, tz);
    if (rc) return rc;
    const int tx = b->tile_x ? b->tile_x : default_xchunk(b, tj, tz);
    const int nmem = (int)b->members.size();
    std::vector<BMember<R>> mem((size_t)nmem);
    std::vector<WorkItem> items;
    std::vector<long long> cost;  // planes per work item
    std::vector<long long> fblk((size_t)nmem + 1, 0);
    for (int i = 0; i < nmem; i++) {
        pf_ctx* c = b->members[(size_t)i];
        BMember<R>& e = mem[(size_t)i];
        memset(&e, 0, sizeof e);
        // view[0]: the level current now; view[1]: after an odd count of steps
        e.view[0] = make_view<R>(c, c->cur, c->old, c->old);
        e.view[1] = make_view<R>(c, c->old, c->cur, c->cur);
        for (Mesh<R>& v : e.view) take_spacings<MODE>(v);
        // planes per chunk: about tx, evened out over the mesh
        const int nch = (c->nx + tx - 1) / tx;
        const int xchunk = std::min((c->nx + nch - 1) / nch, XT - 3);
        e.tm = tile_map(c, tj, tz, xchunk);
        e.step = c->d_step;
        e.t0 = c->step;
        e.budget = c->wave_len;
        const long long nt = (long long)e.tm.nkt * e.tm.njt * e.tm.nxc;
        for (long long t = 0; t < nt; t++) {
            items.push_back({i, (int)t});
            const int xc = (int)(t / ((long long)e.tm.nkt * e.tm.njt));
            const int ib = xc * e.tm.xchunk;
            cost.push_back(std::min(e.tm.xchunk, c->nx - ib) + 2);
        }
        fblk[(size_t)i + 1] = fblk[(size_t)i] + face_blocks(e, c);
    }
    if (items.size() > 0x7fffffff) return fail(PF_ERR_ARG, "batch work-list too long");
    if (fblk[(size_t)nmem] > 0x7fffffffLL) return fail(PF_ERR_ARG, "batch has too many face cells");
    std::vector<FaceBlock> fmap;
    fmap.reserve((size_t)fblk[(size_t)nmem]);
    for (int i = 0; i < nmem; i++)
        for (long long g = fblk[(size_t)i]; g < fblk[(size_t)i + 1]; g++)
            fmap.push_back({i, (int)(g - fblk[(size_t)i])});
    // 8 contiguous runs of (nearly) equal plane count
    long long total = 0;
    for (long long v : cost) total += v;
    std::vector<int> qbeg(NXCD + 1, 0);
    {
        long long acc = 0;
        int q = 1;
        for (size_t t = 0; t < items.size() && q < NXCD; t++) {
            acc += cost[t];
            while (q < NXCD && acc * NXCD >= total * q) qbeg[(size_t)q++] = (int)t + 1;
        }
        while (q < NXCD) qbeg[(size_t)q++] = (int)items.size();
        qbeg[NXCD] = (int)items.size();
    }
    // (re)allocate and upload
    const size_t mb = sizeof(BMember<R>) * (size_t)nmem;
    if (b->mem_bytes < mb || b->items_cap < items.size() || b->fmap_cap < fmap.size() ||
        !b->d_qbeg) {
        free_tables(b);
        HIPCHK(hipMalloc(&b->d_mem, mb));
        HIPCHK(hipMalloc((void**)&b->d_items, sizeof(WorkItem) * std::max<size_t>(items.size(), 1)));
        HIPCHK(hipMalloc((void**)&b->d_qbeg, sizeof(int) * (NXCD + 1)));
        // two steps' queue counters
        HIPCHK(hipMalloc((void**)&b->d_ctr, sizeof(int) * (2 * NXCD)));
        HIPCHK(hipMalloc((void**)&b->d_bstep, sizeof(long long)));
        HIPCHK(hipMalloc((void**)&b->d_fmap, sizeof(FaceBlock) * std::max<size_t>(fmap.size(), 1)));
        b->mem_bytes = mb;
        b->items_cap = std::max<size_t>(items.size(), 1);
        b->fmap_cap = std::max<size_t>(fmap.size(), 1);
    }
    HIPCHK(hipStreamSynchronize(b->stream));
    HIPCHK(hipMemcpy(b->d_mem, mem.data(), mb, hipMemcpyHostToDevice));
    if (!items.empty())
        HIPCHK(hipMemcpy(b->d_items, items.data(), sizeof(WorkItem) * items.size(), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(b->d_qbeg, qbeg.data(), sizeof(int) * (NXCD + 1), hipMemcpyHostToDevice));
    HIPCHK(hipMemset(b->d_ctr, 0, sizeof(int) * (2 * NXCD)));
    HIPCHK(hipMemset(b->d_bstep, 0, sizeof(long long)));
    if (!fmap.empty())
        HIPCHK(hipMemcpy(b->d_fmap, fmap.data(), sizeof(FaceBlock) * fmap.size(), hipMemcpyHostToDevice));
    for (int i = 0; i < nmem; i++) {
        pf_ctx* c = b->members[(size_t)i];
        HIPCHK(hipMemcpy(c->d_step, &c->step, sizeof(long long), hipMemcpyHostToDevice));
    }
    b->face_blocks = fblk[(size_t)nmem];
    if ((rc = free_graph(b))) return rc;
    b->dirty = false;
    return PF_OK;
}

// The FP64 flavour is the one all members allow: reciprocal products, exact
// quotients, else divisions (all the same bits).  16 members of 14.2 M nodes,
// us a step: 286, 355 (at a spacing of 0.3), 399; 5 of 1.4 M: 49, 65, 71.
void choose_mode(pf_batch* b) {
    bool recip = true, quot = true;
    for (const pf_ctx* c : b->members) {
        recip = recip && c->recip;
        quot = quot && c->quot;
    }
    b->mode = b->precision == PF_FP32   ? MODE_FP32
              : b->precision != PF_FP64 ? MODE_FP32C
              : recip                   ? MODE_FP64P
              : quot                    ? MODE_FP64Q
                                        : MODE_FP64;
}

int build(pf_batch* b) {
    choose_mode(b);
    switch (b->mode) {
        case MODE_FP64: return build_t<double, MODE_FP64>(b);
        case MODE_FP64P: return build_t<double, MODE_FP64P>(b);
        case MODE_FP64Q: return build_t<double, MODE_FP64Q>(b);
        case MODE_FP32: return build_t<float, MODE_FP32>(b);
        default: return build_t<float, MODE_FP32C>(b);
    }
}

// Blocks of the sweep with this shape (b->grid).
int shape_grid(pf_batch* b, int tj, int tz) {
    choose_mode(b);
    switch (b->mode) {
        case MODE_FP64: return sweep_grid_t<double, MODE_FP64>(b, tj, tz);
        case MODE_FP64P: return sweep_grid_t<double, MODE_FP64P>(b, tj, tz);
        case MODE_FP64Q: return sweep_grid_t<double, MODE_FP64Q>(b, tj, tz);
        case MODE_FP32: return sweep_grid_t<float, MODE_FP32>(b, tj, tz);
        default: return sweep_grid_t<float, MODE_FP32C>(b, tj, tz);
    }
}

template <class R, int MODE, bool SPONGE, int TJ, int KZ>
void launch_sweep(pf_batch* b, int off) {
    hipLaunchKernelGGL((k_batch_sweep<R, MODE, SPONGE, TJ, KZ>), dim3((unsigned)b->grid), dim3(64, TJ * KZ / 64), 0,
                       b->stream, (const BMember<R>*)b->d_mem, (const WorkItem*)b->d_items, (const int*)b->d_qbeg,
                       b->d_ctr, (const long long*)b->d_bstep, off);
}

template <class R, int MODE, bool SPONGE>
void launch_sweep_s(pf_batch* b, int tj, int tz, int off) {
    if (tz == 64 && tj == 16) launch_sweep<R, MODE, SPONGE, 16, 64>(b, off);
    else if (tz == 64 && tj == 8) launch_sweep<R, MODE, SPONGE, 8, 64>(b, off);
    else if (tz == 32 && tj == 32) launch_sweep<R, MODE, SPONGE, 32, 32>(b, off);
    else if (tz == 32 && tj == 16) launch_sweep<R, MODE, SPONGE, 16, 32>(b, off);
    else launch_sweep<R, MODE, SPONGE, 8, 32>(b, off);
}

// Issue a group of k batched steps on the batch stream: two launches a step
// and the one that moves the counters on.
template <class R, int MODE>
int issue_steps_t(pf_batch* b, int k) {
    int tj, tz;
    batch_shape(b, tj, tz);
    const BMember<R>* mem = (const BMember<R>*)b->d_mem;
    for (int off = 0; off < k; off++) {
        if (b->sponge == 1) launch_sweep_s<R, MODE, true>(b, tj, tz, off);
        else launch_sweep_s<R, MODE, false>(b, tj, tz, off);
        hipLaunchKernelGGL((k_batch_faces<R, face_mode(MODE)>), dim3((unsigned)b->face_blocks), dim3(256), 0, b->stream, mem,
                           (const FaceBlock*)b->d_fmap, (const long long*)b->d_bstep, off);
    }
    hipLaunchKernelGGL((k_batch_advance<R>), dim3(1), dim3(256), 0, b->stream, mem, (int)b->members.size(), b->d_bstep,
                       k);
    HIPCHK(hipGetLastError());
    return PF_OK;
}

int issue_steps(pf_batch* b, int k) {
    switch (b->mode) {
        case MODE_FP64: return issue_steps_t<double, MODE_FP64>(b, k);
        case MODE_FP64P: return issue_steps_t<double, MODE_FP64P>(b, k);
        case MODE_FP64Q: return issue_steps_t<double, MODE_FP64Q>(b, k);
        case MODE_FP32: return issue_steps_t<float, MODE_FP32>(b, k);
        default: return issue_steps_t<float, MODE_FP32C>(b, k);
    }
}

// Capture k steps in a graph (replacing any previous one).
int capture(pf_batch* b, int k) {
    int rc = free_graph(b);
    if (rc) return rc;
    HIPCHK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    rc = issue_steps(b, k);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(b->stream, &g);
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (e != hipSuccess) return fail(PF_ERR_HIP, "graph capture failed: %s", hipGetErrorString(e));
    b->graph = g;
    HIPCHK(hipGraphInstantiate(&b->exec, g, nullptr, nullptr, 0));
    b->graph_steps = k;
    return PF_OK;
}

// Steps each member takes of the next n batched steps, and its new state.
void account(pf_batch* b, long long n) {
    for (pf_ctx* c : b->members) {
        const long long left = c->wave_len - c->step;
        const long long take = n < left ? n : (left > 0 ? left : 0);
        c->step += take;
        if (take & 1) {
            const int t = c->cur;
            c->cur = c->old;
            c->old = t;
        }
    }
}

constexpr int GRAPH_STEPS = 16;

int step_n(pf_batch* b, long long n) {
    int rc;
    if (b->dirty && (rc = build(b))) return rc;
    long long done = 0;
    if (b->use_graph && n >= GRAPH_STEPS) {
        if (b->graph_steps != GRAPH_STEPS && (rc = capture(b, GRAPH_STEPS))) return rc;
        for (; done + GRAPH_STEPS <= n; done += GRAPH_STEPS) HIPCHK(hipGraphLaunch(b->exec, b->stream));
    }
    for (; done < n; done += std::min<long long>(n - done, GRAPH_STEPS))
        if ((rc = issue_steps(b, (int)std::min<long long>(n - done, GRAPH_STEPS)))) return rc;
    account(b, n);
    return PF_OK;
}

}  // namespace

// ------------------------------------------------------------ C ABI ----
extern "C" int pf_batch_create(int32_t precision, pf_batch** out) {
    if (!out) return fail(PF_ERR_ARG, "out is NULL");
    *out = nullptr;
    if (precision < PF_FP64 || precision > PF_FP32C) return fail(PF_ERR_ARG, "bad precision %d", precision);
    pf_batch* b = new (std::nothrow) pf_batch();
    if (!b) return fail(PF_ERR_NOMEM, "out of host memory");
    b->precision = precision;
    int rc = PF_OK;
    if (hipGetDevice(&b->dev) != hipSuccess ||
        hipDeviceGetAttribute(&b->cus, hipDeviceAttributeMultiprocessorCount, b->dev) != hipSuccess ||
        hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess)
        rc = fail(PF_ERR_HIP, "batch stream creation failed");
    if (rc) {
        delete b;
        return rc;
    }
    *out = b;
    return PF_OK;
}

extern "C" int pf_batch_add(pf_batch* b, pf_ctx* c) {
    if (!b || !c) return fail(PF_ERR_ARG, "NULL argument");
    if (c->batch) return fail(PF_ERR_STATE, "context is already in a batch");
    if (c->precision != b->precision) return fail(PF_ERR_ARG, "context precision %d != batch precision %d", c->precision, b->precision);
    if (c->nmat > PF_TILED_MAX_MATERIALS)
        return fail(PF_ERR_ARG, "batched sweeps hold at most %d materials (got %d)", PF_TILED_MAX_MATERIALS, c->nmat);
    if (level_bytes(c->cells, c->precision) >= (1ULL << 32))
        return fail(PF_ERR_ARG, "a batch member's time level must be < 4 GiB");
    const int sp = c->sponge ? 1 : 0;
    if (!b->members.empty() && b->sponge != sp)
        return fail(PF_ERR_ARG, "all members of a batch either have an absorbing layer or none");
    HIPCHK(hipStreamSynchronize(c->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    take_quotients(c);
    b->sponge = sp;
    b->members.push_back(c);
    c->batch = b;
    c->batch_stream = b->stream;
    b->dirty = true;
    return PF_OK;
}

extern "C" int pf_batch_remove(pf_batch* b, pf_ctx* c) {
    if (!b || !c) return fail(PF_ERR_ARG, "NULL argument");
    auto it = std::find(b->members.begin(), b->members.end(), c);
    if (it == b->members.end()) return fail(PF_ERR_STATE, "context is not a member of this batch");
    HIPCHK(hipStreamSynchronize(b->stream));
    b->members.erase(it);
    c->batch = nullptr;
    c->batch_stream = nullptr;
    b->dirty = true;
    return PF_OK;
}

extern "C" int pf_batch_step(pf_batch* b, int64_t nsteps) {
    if (!b) return fail(PF_ERR_ARG, "batch is NULL");
    if (nsteps < 0) return fail(PF_ERR_ARG, "nsteps < 0");
    if (b->members.empty() || nsteps == 0) return PF_OK;
    return step_n(b, nsteps);
}

extern "C" int pf_batch_sync(pf_batch* b) {
    if (!b) return fail(PF_ERR_ARG, "batch is NULL");
    HIPCHK(hipStreamSynchronize(b->stream));
    return PF_OK;
}

extern "C" int pf_batch_set_tiles(pf_batch* b, int32_t tile_j, int32_t tile_z, int32_t tile_x, int32_t use_graph) {
    if (!b) return fail(PF_ERR_ARG, "batch is NULL");
    int tj = tile_j, tz = tile_z;
    resolve_shape(b->precision, 0, tj, tz);
    if (!shape_built(tj, tz)) return fail(PF_ERR_ARG, "batch tile shape %d rows x %d lanes is not built", tj, tz);
    if (tile_x < 0 || tile_x > XT - 3) return fail(PF_ERR_ARG, "tile_x must be 0..%d", XT - 3);
    HIPCHK(hipStreamSynchronize(b->stream));
    b->tile_j = tile_j;
    b->tile_z = tile_z;
    b->tile_x = tile_x;
    b->use_graph = use_graph != 0;
    b->dirty = true;
    return PF_OK;
}

extern "C" int pf_batch_autotune(pf_batch* b, int32_t trial_steps, int32_t* tile_j, int32_t* tile_z, int32_t* tile_x,
                                 double* ms_per_step) {
    if (!b) return fail(PF_ERR_ARG, "batch is NULL");
    if (trial_steps < 1) return fail(PF_ERR_ARG, "trial_steps < 1");
    if (b->members.empty()) return fail(PF_ERR_STATE, "batch has no members");
    struct Cand { int tj, tz, tx; };
    std::vector<Cand> cands;
    const int shapes[][2] = {{16, 64}, {8, 64}, {32, 32}, {16, 32}, {8, 32}};
    const int shapes64[][2] = {{8, 32}, {16, 32}, {8, 64}};
    const bool f64 = b->precision == PF_FP64;
    for (int q = 0; q < (f64 ? 3 : 5); q++) {
        const int* const sh = f64 ? shapes64[q] : shapes[q];
        // the shape's default chunk among them: below 32 planes, where it is
        // none of the others, it takes the place of 128, whose items would
        // leave most blocks without one
        int rc = shape_grid(b, sh[0], sh[1]);
        if (rc) return rc;
        const int own = default_xchunk(b, sh[0], sh[1]);
        for (int tx : {16, 32, 64, own == 16 || own == 32 ? 128 : own}) cands.push_back({sh[0], sh[1], tx});
    }
    // every candidate runs 1 untimed + trial_steps timed steps of real work
    long long room = 0;
    for (pf_ctx* c : b->members) room = std::max(room, c->wave_len - c->step);
    if (room < (long long)cands.size() * (trial_steps + 1))
        return fail(PF_ERR_RANGE, "members have %lld steps left; autotuning needs %lld", room,
                    (long long)cands.size() * (trial_steps + 1));
    const int keep_j = b->tile_j, keep_z = b->tile_z, keep_x = b->tile_x;
    const bool keep_g = b->use_graph;
    double best = 1e300;
    Cand bc = cands[0];
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreateWithFlags(&e0, PF_TIMING_EVENT));
    HIPCHK(hipEventCreateWithFlags(&e1, PF_TIMING_EVENT));
    int rc = PF_OK;
    for (const Cand& k : cands) {
        b->tile_j = k.tj; b->tile_z = k.tz; b->tile_x = k.tx;
        b->use_graph = false;
        b->dirty = true;
        if ((rc = step_n(b, 1))) break;  // builds the tables, warms the kernel
        if (hipEventRecord(e0, b->stream) != hipSuccess) { rc = fail(PF_ERR_HIP, "event record"); break; }
        if ((rc = step_n(b, trial_steps))) break;
        if (hipEventRecord(e1, b->stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess) {
            rc = fail(PF_ERR_HIP, "event sync");
            break;
        }
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, e0, e1);
        const double per = ms / trial_steps;
        if (per < best) { best = per; bc = k; }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) {
        b->tile_j = keep_j; b->tile_z = keep_z; b->tile_x = keep_x;
        b->use_graph = keep_g;
        b->dirty = true;
        return rc;
    }
    b->tile_j = bc.tj; b->tile_z = bc.tz; b->tile_x = bc.tx;
    b->use_graph = keep_g;
    b->dirty = true;
    if (tile_j) *tile_j = bc.tj;
    if (tile_z) *tile_z = bc.tz;
    if (tile_x) *tile_x = bc.tx;
    if (ms_per_step) *ms_per_step = best;
    return PF_OK;
}

extern "C" int pf_batch_destroy(pf_batch* b) {
    if (!b) return PF_OK;
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    for (pf_ctx* c : b->members) {
        c->batch = nullptr;
        c->batch_stream = nullptr;
    }
    (void)free_graph(b);
    free_tables(b);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
    return PF_OK;
}
