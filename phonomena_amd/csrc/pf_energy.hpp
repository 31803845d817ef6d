// Energy audit kernels: E = dV/2 [ sum rho_q ((u_q - u_q_old)/dt)^2
//                                 + sum over stress sites of T(u) : strain(u_old) ],
// the quantity the leapfrog scheme conserves, in FP64 from the two newest
// levels as stored (FP32 values widened, lo parts added).
//
// A thread takes one (y, z) cell of the planes of an x chunk.  It keeps the
// plane's and the next plane's own values in registers; the neighbours along
// z are lane shifts (a wave's outer lanes repeat its neighbours' cells), those
// along y loads that hit the lines the next row's own values bring in, so a
// level is read from HBM once.  Strains are formed once per level and site
// with reciprocal spacings (1 ulp from a quotient; the FP64 divisions they
// replace, thirty a node, were most of the kernel's time), stresses from the
// newest level's.  Bound: instructions and the waves in flight (122 VGPRs, 146
// in FP32C).  A call on 257 x 257 x 129 nodes takes 128 us in FP32C, 83 in
// FP32, 130 in FP64 (166, 95 and 150 with the z neighbours loaded and decoded
// again), against 680, 621 and 453 with levels widened to FP64 arrays by
// six launches first and a grid-stride kernel with 64-bit index divisions and
// quotients per node; 21 us on small meshes (81 in FP32C, 42 in FP64).  A
// context's first call costs 3 us more: the partial sums are allocated with it
// and the two sums pass through the transfers' pinned memory (allocated by the
// first call they cost 26 to 40 us there).  The relative error against a
// 64-bit restatement is the same (2e-16 to 8e-16 in FP64).
//
// Per-thread sums, a wavefront/LDS tree per block, then one block adds the
// block partials in a fixed order, so the result is deterministic.
#pragma once
#include "pf_tiled.hpp"

namespace pf {

struct EnergyArgs {
    const double* mat;         // rows of the FP64 material table
    const double* rho;         // density per material
    const double *fx, *fy, *fz, *sx, *sy, *sz;  // FP64 spacings
    double f0[3], s0[3];       // first spacings
    double dt;
    const double* w_prev;      // source of the step that produced the newest level (null: none)
    int xchunk;                // planes per block
    unsigned per;              // blocks per chunk: block b takes cells ENERGY_CELLS (b % per) ... of chunk b / per
};

PF_DEV double warp_sum(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

constexpr int ENERGY_XCHUNK = 32;  // most planes per block
constexpr int ENERGY_CELLS = 4 * 62;  // cells per block: a wave's outer lanes are its neighbours' cells

// About 8 blocks per CU, 4 to ENERGY_XCHUNK planes each.
inline EnergyGrid energy_grid(int nx, long long plane) {
    EnergyGrid g;
    g.per = (plane + ENERGY_CELLS - 1) / ENERGY_CELLS;
    long long want = (2048 + g.per - 1) / g.per;
    if (want > (nx + 3) / 4) want = (nx + 3) / 4;
    g.xchunk = (int)((nx + want - 1) / want);
    if (g.xchunk > ENERGY_XCHUNK) g.xchunk = ENERGY_XCHUNK;
    g.blocks = g.per * ((nx + g.xchunk - 1) / g.xchunk);
    return g;
}

// One level's value of a component at cell a of its array.
template <bool COMP, class R>
PF_DEV double energy_at(const R* __restrict__ h, const lo_t* __restrict__ l, long long a) {
    const R v = h[a];
    if constexpr (COMP) return (double)v + (double)lo_decode(v, l[a]);
    return (double)v;
}

// The strains of one level at a node's sites: normal e1..e3, brackets of
// T4..T6.  Own values of plane i (x, y, z), ux of plane i-1, uy and uz of
// plane i+1, and the y and z neighbours of plane i.
struct Strain {
    double e1, e2, e3, g4, g5, g6;
};

// m: c* = newest level, o* = previous level.  As in the reference's arrays
// after time_step, the previous level carries the source value on its uz
// wall line (u_old was copied after the source write) and the newest level
// carries what the step stored there.
template <class R, bool COMP>
__global__ __launch_bounds__(256) void k_energy_partial(Mesh<R> m, EnergyArgs ea, double* __restrict__ partials) {
    extern __shared__ double smat[];  // material rows, then densities
    __shared__ double rx[ENERGY_XCHUNK][2];  // 1 / sx, 1 / fx of the chunk's planes
    __shared__ double red[2][4];
    const int i0 = (int)(blockIdx.x / ea.per) * ea.xchunk, i1 = min(i0 + ea.xchunk, m.nx);
    for (int e = threadIdx.x; e < m.nmat * MAT_STRIDE; e += 256) smat[e] = ea.mat[e];
    double* const srho = smat + m.nmat * MAT_STRIDE;
    for (int e = threadIdx.x; e < m.nmat; e += 256) srho[e] = ea.rho[e];
    if ((int)threadIdx.x < i1 - i0) {
        const int i = i0 + (int)threadIdx.x;
        rx[threadIdx.x][0] = i >= 1 && i <= m.nx - 2 ? 1.0 / ea.sx[i - 1] : 0.0;
        rx[threadIdx.x][1] = i <= m.nx - 2 ? 1.0 / ea.fx[i] : 0.0;
    }
    __syncthreads();
    double ke = 0.0, se = 0.0;
    const long long plane = m.plane;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    // cells before the plane's first and past its last take those (and, as
    // every outer lane, add nothing)
    long long t = (long long)(blockIdx.x % ea.per) * ENERGY_CELLS + wv * 62 + lane - 1;
    const bool own = lane >= 1 && lane <= 62 && t < plane;
    t = t < 0 ? 0 : (t < plane ? t : plane - 1);
    {
        const int j = (int)(t / m.pz), k = (int)(t % m.pz);
        const bool ks = k >= 1, kf = k <= m.nz - 2, jn = j >= 1 && j <= m.ny - 2, jf = j <= m.ny - 2;
        // k = 0 takes the first spacings, in the reference's order (as the
        // column constants of the sweeps)
        const double rfx0 = 1.0 / ea.f0[0], rfy0 = 1.0 / ea.f0[1], rfz0 = 1.0 / ea.f0[2];
        const double rfy = jf ? 1.0 / ea.fy[j] : 0.0, rfz = kf ? 1.0 / ea.fz[k] : 0.0;
        const double ry = !ks ? 1.0 / ea.s0[1] : jn ? 1.0 / ea.sy[j - 1] : 0.0;
        const double rz = !ks ? 1.0 / ea.s0[2] : kf ? 1.0 / ea.sz[k - 1] : 0.0;
        const double rsx0 = 1.0 / ea.s0[0], rdt = 1.0 / ea.dt;
        const double h41 = ks ? rfz : rfy0, h42 = ks ? rfy : rfz0, h51 = ks ? rfz : rfx0, h61 = ks ? rfy : rfx0;
        const double wp = ea.w_prev && k == 0 && i0 == 0 ? *ea.w_prev : 0.0;
        // neighbours inside the plane: along y cells without one read
        // themselves, along z the lanes beside take the next row's; their
        // terms are left out
        const long long jp = jf ? m.pz : 0, jm = j >= 1 ? m.pz : 0, kp = k <= m.nz - 2 ? 1 : 0;
        const long long kq = ks ? kp : 0;
        long long a = (long long)i0 * plane + t;
        // own values: [level][component], planes i and i+1, ux of plane i-1
        double u[2][3], un[2][3], uxm[2];
        const long long am = i0 >= 1 ? a - plane : a;
        u[0][0] = energy_at<COMP>(m.c0, m.cl0, a);
        u[0][1] = energy_at<COMP>(m.c1, m.cl1, a);
        u[0][2] = energy_at<COMP>(m.c2, m.cl2, a);
        u[1][0] = energy_at<COMP>(m.o0, m.ol0, a);
        u[1][1] = energy_at<COMP>(m.o1, m.ol1, a);
        u[1][2] = energy_at<COMP>(m.o2, m.ol2, a);
        uxm[0] = energy_at<COMP>(m.c0, m.cl0, am);
        uxm[1] = energy_at<COMP>(m.o0, m.ol0, am);
        int id = m.ids[a], id_j = m.ids[a + jp], id_k = m.ids[a + kp];
        for (int i = i0; i < i1; i++, a += plane) {
            const long long an = i <= m.nx - 2 ? a + plane : a;
            un[0][0] = energy_at<COMP>(m.c0, m.cl0, an);
            un[0][1] = energy_at<COMP>(m.c1, m.cl1, an);
            un[0][2] = energy_at<COMP>(m.c2, m.cl2, an);
            un[1][0] = energy_at<COMP>(m.o0, m.ol0, an);
            un[1][1] = energy_at<COMP>(m.o1, m.ol1, an);
            un[1][2] = energy_at<COMP>(m.o2, m.ol2, an);
            const int in = m.ids[an], in_j = m.ids[an + jp], in_k = m.ids[an + kp], id_jk = m.ids[a + jp + kq];
            const bool ii = i <= m.nx - 2, is = i >= 1 && ii;
            const double rsx = ks ? rx[i - i0][0] : rsx0, rfx = rx[i - i0][1], h52 = ks ? rfx : rfz0;
            Strain s[2];
#pragma unroll
            for (int l = 0; l < 2; l++) {
                const R* const h0 = l ? m.o0 : m.c0;
                const R* const h1 = l ? m.o1 : m.c1;
                const R* const h2 = l ? m.o2 : m.c2;
                const lo_t* const l0 = l ? m.ol0 : m.cl0;
                const lo_t* const l1 = l ? m.ol1 : m.cl1;
                const lo_t* const l2 = l ? m.ol2 : m.cl2;
                const bool sub = l && i == 0 && k == 0 && ea.w_prev;
                const double z = sub ? wp : u[l][2];
                const double zj = sub ? wp : energy_at<COMP>(h2, l2, a + jp);
                const double zb = below0(u[l][2]), zm = ks ? zb : 0.0;
                s[l].e1 = (u[l][0] - uxm[l]) * rsx;
                s[l].e2 = (u[l][1] - energy_at<COMP>(h1, l1, a - jm)) * ry;
                s[l].e3 = (z - zm) * rz;
                s[l].g4 = (above0(u[l][1]) - u[l][1]) * h41 + (zj - z) * h42;
                s[l].g5 = (above0(u[l][0]) - u[l][0]) * h51 + (un[l][2] - z) * h52;
                s[l].g6 = (energy_at<COMP>(h0, l0, a + jp) - u[l][0]) * h61 + (un[l][1] - u[l][1]) * h52;
            }
            if (is && jn && kf) {
                const double* c = smat + id * MAT_STRIDE;
                const double t1 = c[M_C00] * s[0].e1 + c[M_C01] * s[0].e2 + c[M_C02] * s[0].e3;
                const double t2 = c[M_C10] * s[0].e1 + c[M_C11] * s[0].e2 + c[M_C12] * s[0].e3;
                const double t3 = c[M_C20] * s[0].e1 + c[M_C21] * s[0].e2 + c[M_C22] * s[0].e3;
                se += t1 * s[1].e1 + t2 * s[1].e2 + (ks ? t3 * s[1].e3 : 0.0);
            }
            if (is && jf && kf) se += (smat[id_jk * MAT_STRIDE + M_C33] * s[0].g4) * s[1].g4;
            if (ii && jn && kf) se += (smat[(ks ? in_k : in) * MAT_STRIDE + M_C44] * s[0].g5) * s[1].g5;
            if (ii && jf && kf) se += (smat[in_j * MAT_STRIDE + M_C55] * s[0].g6) * s[1].g6;
            // kinetic terms; the x = 0 wall of uy (clamped) and uz (driven) is left out
            if (ii) {
                const double v = (u[0][0] - u[1][0]) * rdt;
                ke += srho[in] * (v * v);
            }
            if (i >= 1 && jf) {
                const double v = (u[0][1] - u[1][1]) * rdt;
                ke += srho[id_j] * (v * v);
            }
            if (i >= 1 && kf) {
                const double v = (u[0][2] - u[1][2]) * rdt;
                ke += srho[id_k] * (v * v);
            }
#pragma unroll
            for (int l = 0; l < 2; l++) {
                uxm[l] = u[l][0];
#pragma unroll
                for (int q = 0; q < 3; q++) u[l][q] = un[l][q];
            }
            id = in;
            id_j = in_j;
            id_k = in_k;
        }
    }
    ke = warp_sum(own ? ke : 0.0);
    se = warp_sum(own ? se : 0.0);
    if (lane == 0) { red[0][wv] = ke; red[1][wv] = se; }
    __syncthreads();
    if (threadIdx.x == 0) {
        const long long b = blockIdx.x;
        partials[2 * b] = ((red[0][0] + red[0][1]) + red[0][2]) + red[0][3];
        partials[2 * b + 1] = ((red[1][0] + red[1][1]) + red[1][2]) + red[1][3];
    }
}

static __global__ __launch_bounds__(1024) void k_energy_final(const double* __restrict__ partials, long long nblk,
                                                       double* __restrict__ out) {
    __shared__ double red[2][1024];
    double ke = 0.0, se = 0.0;
    for (long long b = threadIdx.x; b < nblk; b += 1024) {
        ke += partials[2 * b];
        se += partials[2 * b + 1];
    }
    red[0][threadIdx.x] = ke;
    red[1][threadIdx.x] = se;
    __syncthreads();
    for (int s = 512; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            red[0][threadIdx.x] += red[0][threadIdx.x + s];
            red[1][threadIdx.x] += red[1][threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) { out[0] = red[0][0]; out[1] = red[1][0]; }
}

}  // namespace pf
