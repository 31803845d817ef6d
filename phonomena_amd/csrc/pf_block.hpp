// Whole steps of a small mesh, several per launch, one thread per node.
//
// The tiled march runs a block's planes one after another (0.7 us a plane in
// FP32, 1.6 us in FP64 with divisions, when a CU holds one block) and needs a
// face launch per step: on meshes too small to fill the chip a step is that
// chain, not its arithmetic or its bytes.  Here a block owns a box of nodes
// and takes T whole steps of them (stresses, update, Mur faces, source,
// probes) in one launch: it loads the box and T more nodes on every side
// that is not the mesh's own, keeps both levels of a node in its thread's
// registers, exchanges displacements and stresses through LDS, and stores
// the owned nodes of the last two levels.  Every step one more ring of the
// box goes stale (its outer neighbours are missing); after T steps what is
// left is exactly the owned box.  No block waits for another: the levels
// read and the levels written are different buffers (for T = 1 the previous
// level, which only its own node reads, is written in place).
//
// What bounds it: the launch (about 4 us with its loads and stores) and the
// chain of T steps; block_map weighs the nodes computed twice against the
// launches saved.  The faces take a pass per axis over values in LDS; as a
// recursion over the faces a cell lies on they cost twice the step (one step of
// 31 x 21 x 6 nodes in FP64 with divisions 9.9 against 7.4 us a launch).
//
// The values are those of the sweep and the face kernels, bit for bit: the
// shared formulas with the same operands, lo parts rounded to their storage
// after every step, z = max faces from the unrounded value below, x and y
// faces and the box edges in the reference's order from values as stored.
#pragma once
#include "pf_tiled.hpp"

namespace pf {

constexpr int BLOCK_MAX_NODES = 1024;    // threads of a block: nodes of its box with halo

// Displacement and stress values of a block's nodes, in dynamic LDS: arrays
// of `threads` values each, u (hi), then in FP32C u (lo), then T1..T6.  T1..T6
// also take the new level between the update and the faces.
template <class R, bool COMP>
PF_DEV R* block_u(R* s, int n, int q) { return s + (size_t)q * n; }
template <class R, bool COMP>
PF_DEV R* block_ul(R* s, int n, int q) { return s + (size_t)(3 + q) * n; }
template <class R, bool COMP>
PF_DEV R* block_t(R* s, int n, int q) { return s + (size_t)((COMP ? 6 : 3) + q) * n; }
template <class R, int MODE>
constexpr size_t block_lds(int threads) {
    return sizeof(R) * (size_t)threads * (MODE == MODE_FP32C ? 12 : 9);
}

// A component's value of one level at the thread's node: hi, lo as decoded
// from its storage, and the stored lo.
template <class R>
struct Own {
    R h, l;
    lo_t q;
};
template <int MODE, class R>
PF_DEV Own<R> block_load(const R* h, const lo_t* l, long long id) {
    Own<R> o;
    o.h = h[id];
    o.q = MODE == MODE_FP32C ? l[id] : (lo_t)0;
    o.l = MODE == MODE_FP32C ? lo_decode(o.h, o.q) : R(0);
    return o;
}
template <int MODE, class R>
PF_DEV Own<R> block_stored(V<R> v) {
    Own<R> o;
    o.h = v.h;
    o.q = MODE == MODE_FP32C ? lo_encode(v.h, v.l) : (lo_t)0;
    o.l = MODE == MODE_FP32C ? lo_decode(v.h, o.q) : R(0);
    return o;
}
template <int MODE, class R>
PF_DEV void block_put(R* h, lo_t* l, long long id, const Own<R>& o) {
    h[id] = o.h;
    if constexpr (MODE == MODE_FP32C) l[id] = o.q;
}

// Where a component's cell stands: none of its cells, a stage-I cell, or the
// face that writes it last (base_solver.py:539-554; of the cells below
// z = max the x face those with 0 < j < Ly, the y faces the others).
enum : int { CELL_NONE = 0, CELL_IN, CELL_X, CELL_Y0, CELL_Y1, CELL_Z };
template <int Q, class R>
PF_DEV int cell_kind(const Mesh<R>& m, int i, int j, int k) {
    const int Lx = Ext<Q>::Lx(m.nx), Ly = Ext<Q>::Ly(m.ny), Lz = Ext<Q>::Lz(m.nz);
    if (i > Lx || j > Ly || k > Lz) return CELL_NONE;
    if (k == Lz) return CELL_Z;
    return j == 0 ? CELL_Y0 : j == Ly ? CELL_Y1 : i == Lx ? CELL_X : CELL_IN;
}
// Whether the cell's column (all k) is one of an x or y face.
template <int Q, class R>
PF_DEV bool face_column(const Mesh<R>& m, int i, int j) {
    return i == Ext<Q>::Lx(m.nx) || j == 0 || j == Ext<Q>::Ly(m.ny);
}

// `steps` whole steps of every node.  m: the view of the first step, levels
// n (c*, cl*) and n-1 (o*, ol*); n* take level n+steps and, for steps > 1,
// p* level n+steps-1.
template <class R, int MODE, bool SPONGE, int MOST>
__global__ __launch_bounds__(MOST) void k_block_steps(Mesh<R> m, R* p0, R* p1, R* p2, lo_t* pl0, lo_t* pl1, lo_t* pl2,
                                                      BlockMap bm, int steps, FaceProbe pr) {
    constexpr int EXACT = exact_of(MODE);
    constexpr bool COMP = MODE == MODE_FP32C;
    extern __shared__ char block_lds_raw[];
    R* const s = (R*)block_lds_raw;
    __shared__ R smat[PF_TILED_MAX_MATERIALS * MAT_STRIDE];
    const int n = (int)blockDim.x, tid = (int)threadIdx.x;
    const long long tt0 = m.step_off;

    // the block's box: owned nodes a0 .. a1-1, with halo i0 .. i1-1
    int b = xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const int bz = b % bm.ntz;
    b /= bm.ntz;
    const int by = b % bm.nty, bx = b / bm.nty;
    const int ax0 = bx * m.nx / bm.ntx, ax1 = (bx + 1) * m.nx / bm.ntx;
    const int ay0 = by * m.ny / bm.nty, ay1 = (by + 1) * m.ny / bm.nty;
    const int az0 = bz * m.nz / bm.ntz, az1 = (bz + 1) * m.nz / bm.ntz;
    const int i0 = max(ax0 - steps, 0), i1 = min(ax1 + steps, m.nx);
    const int j0 = max(ay0 - steps, 0), j1 = min(ay1 + steps, m.ny);
    const int k0 = max(az0 - steps, 0), k1 = min(az1 + steps, m.nz);
    const int ey = j1 - j0, ez = k1 - k0, nodes = (i1 - i0) * ey * ez;
    const bool active = tid < nodes;
    const int k = k0 + tid % ez, j = j0 + tid / ez % ey, i = i0 + min(tid / (ez * ey), i1 - i0 - 1);
    // whether the box holds cells of a face (uniform over the block)
    const bool faces = j0 == 0 || j1 >= m.ny - 1 || i1 >= m.nx - 1 || k1 >= m.nz - 1;

    for (int e = tid; e < m.nmat * MAT_STRIDE; e += n) smat[e] = m.mat[e];

    // levels n and n-1 of the node (n-1 beside the owned nodes only where a
    // later step needs it: for one step its owner writes it in place)
    const bool own = active && i >= ax0 && i < ax1 && j >= ay0 && j < ay1 && k >= az0 && k < az1;
    const long long id = at(m, i, j, k);
    const bool src = i == 0 && k == 0;
    Own<R> c0 = block_load<MODE>(m.c0, m.cl0, id), c1 = block_load<MODE>(m.c1, m.cl1, id),
           c2 = block_load<MODE>(m.c2, m.cl2, id);
    const Own<R> zero = {R(0), R(0), (lo_t)0};
    Own<R> q0 = zero, q1 = zero, q2 = zero;
    if (own || steps > 1) {
        q0 = block_load<MODE>(m.o0, m.ol0, id);
        q1 = block_load<MODE>(m.o1, m.ol1, id);
        q2 = block_load<MODE>(m.o2, m.ol2, id);
    }
    // material of the node and of the nodes its values are sampled at
    const int ip = min(i + 1, m.nx - 1), jp = min(j + 1, m.ny - 1), kp = min(k + 1, m.nz - 1);
    const bool ks = k >= 1;
    const int kq = ks ? kp : k;
    const int id_c = m.ids[id], id_4 = m.ids[at(m, i, jp, kq)], id_5 = m.ids[at(m, ip, j, kq)],
              id_6 = m.ids[at(m, ip, jp, k)], id_x = m.ids[at(m, ip, j, k)], id_y = m.ids[at(m, i, jp, k)],
              id_z = m.ids[at(m, i, j, kq)];

    // column constants, as in the tiled march
    const bool in = i >= 1 && i <= m.nx - 2, ih = i <= m.nx - 2;
    const bool jn = j >= 1 && j <= m.ny - 2, jf = j <= m.ny - 2;
    const bool kf = k <= m.nz - 2;
    const R hsx = in ? m.sx[i - 1] : R(1), hfx = ih ? m.fx[i] : R(1);
    const R hsy = jn ? m.sy[j - 1] : R(1), hfy = jf ? m.fy[j] : R(1);
    const R hsz = ks && kf ? m.sz[k - 1] : R(1), hfz = kf ? m.fz[k] : R(1);
    const R hx_n = sel(ks, hsx, m.sx0), hx_f = sel(ks, hfx, m.fx0), fxi = sel(ks, hfx, m.fz0);
    const R hy_n = sel(ks, hsy, m.sy0), hz_n = sel(ks, hsz, m.sz0);
    const R s4_h1 = sel(ks, hfz, m.fy0), s4_h2 = sel(ks, hfy, m.fz0);
    const R s5_h1 = sel(ks, hfz, m.fx0), s6_h1 = sel(ks, hfy, m.fx0);
    const R uy_g2 = sel(ks, hfy, m.fy0);
    const R uz_g3 = sel(ks || m.surf, hfz, R(1));
    const R damp = SPONGE ? (m.dpx[i] + m.dpy[j]) + m.dpz[k] : R(0);
    const bool nv = in && jn && kf;
    // neighbours in the box (a node without one keeps itself: what it then
    // computes is masked, a cell of a face, or in a stale ring)
    const int dx = ey * ez;
    const int t = min(tid, nodes - 1);  // idle threads stand on the last node and store nothing
    const int xm = active && i > i0 ? t - dx : t, xp = active && i < i1 - 1 ? t + dx : t;
    const int ym = active && j > j0 ? t - ez : t, yp = active && j < j1 - 1 ? t + ez : t;
    const int zm = active && k > k0 ? t - 1 : t, zp = active && k < k1 - 1 ? t + 1 : t;
    const int kind0 = cell_kind<0>(m, i, j, k), kind1 = cell_kind<1>(m, i, j, k), kind2 = cell_kind<2>(m, i, j, k);
    R* const u0 = block_u<R, COMP>(s, n, 0);
    R* const u1 = block_u<R, COMP>(s, n, 1);
    R* const u2 = block_u<R, COMP>(s, n, 2);
    R* const t1 = block_t<R, COMP>(s, n, 0);
    R* const t2 = block_t<R, COMP>(s, n, 1);
    R* const t3 = block_t<R, COMP>(s, n, 2);
    R* const t4 = block_t<R, COMP>(s, n, 3);
    R* const t5 = block_t<R, COMP>(s, n, 4);
    R* const t6 = block_t<R, COMP>(s, n, 5);

    // the current level into LDS, with the source value of step tt on the
    // wall line; c2 keeps the stored value
    Own<R> w2 = c2;
    auto publish = [&](long long tt) {
        w2 = c2;
        if (src) w2 = {(R)m.wave[tt], R(0), (lo_t)0};
        if (active) {
            u0[tid] = c0.h;
            u1[tid] = c1.h;
            u2[tid] = w2.h;
            if constexpr (COMP) {
                block_ul<R, COMP>(s, n, 0)[tid] = c0.l;
                block_ul<R, COMP>(s, n, 1)[tid] = c1.l;
                block_ul<R, COMP>(s, n, 2)[tid] = w2.l;
            }
        }
    };
    publish(tt0);

    for (int r = 0; r < steps; r++) {
        __syncthreads();
        // stresses (base_solver.py:329-372, 408-433)
        R n1, n2, n3;
        normal3<EXACT>(smat + id_c * MAT_STRIDE, c0.h - u0[xm], c1.h - u1[ym], w2.h - sel(ks, u2[zm], R(0)), hx_n, hy_n,
                       hz_n, n1, n2, n3);
        n1 = sel(nv, n1, R(0));
        n2 = sel(nv, n2, R(0));
        n3 = sel(nv && ks, n3, R(0));
        R s4 = shear<EXACT>(smat[id_4 * MAT_STRIDE + M_C33], u1[zp] - c1.h, s4_h1, u2[yp] - w2.h, s4_h2);
        R s5 = shear<EXACT>(smat[id_5 * MAT_STRIDE + M_C44], u0[zp] - c0.h, s5_h1, u2[xp] - w2.h, fxi);
        R s6 = shear<EXACT>(smat[id_6 * MAT_STRIDE + M_C55], u0[yp] - c0.h, s6_h1, u1[xp] - c1.h, fxi);
        s4 = sel(in && jf && kf, s4, R(0));
        s5 = sel(ih && jn && kf, s5, R(0));
        s6 = sel(ih && jf && kf, s6, R(0));
        if (active) {
            t1[tid] = n1;
            t2[tid] = n2;
            t3[tid] = n3;
            t4[tid] = s4;
            t5[tid] = s5;
            t6[tid] = s6;
        }
        __syncthreads();
        // update (base_solver.py:441-463, 495-517)
        V<R> a0, a1, a2;
        {
            const R dv = div3<EXACT>(t1[xp] - n1, hx_f, s6 - t6[ym], hy_n, s5 - sel(ks, t5[zm], R(0)), hz_n);
            a0 = leap_from<MODE, SPONGE>(V<R>{c0.h, c0.l}, q0.h, q0.l, smat[id_x * MAT_STRIDE + M_COEF], dv, damp);
        }
        {
            const R dv = div3<EXACT>(s6 - t6[xm], hx_n, t2[yp] - n2, uy_g2, s4 - sel(ks, t4[zm], R(0)), hz_n);
            a1 = leap_from<MODE, SPONGE>(V<R>{c1.h, c1.l}, q1.h, q1.l, smat[id_y * MAT_STRIDE + M_COEF], dv, damp);
        }
        {
            const R dv = div3<EXACT>(s5 - t5[xm], hx_n, s4 - t4[ym], hy_n, t3[zp] - n3, uz_g3);
            a2 = leap_from<MODE, SPONGE>(V<R>{w2.h, w2.l}, q2.h, q2.l, smat[id_z * MAT_STRIDE + M_COEF], dv, damp);
        }
        if (i == 0) a1 = a2 = {R(0), R(0)};  // uy, uz on the x = 0 wall stay 0
        if (faces) {
            // The stage-I values as stored go to LDS (T1..T6 are done with),
            // and the z = max faces off the x and y faces with them, mapped
            // from the value below before it is rounded.  Then the faces in
            // the reference's order, a pass each: x, y (both), z, every map
            // reading the cell one inside as the passes before it left it.
            const Own<R> g0 = block_stored<MODE>(a0), g1 = block_stored<MODE>(a1), g2 = block_stored<MODE>(a2);
            __syncthreads();
            auto level = [&](auto Qc, int at) {
                constexpr int Q = decltype(Qc)::value;
                return V<R>{block_u<R, COMP>(s, n, Q)[at], COMP ? block_ul<R, COMP>(s, n, Q)[at] : R(0)};
            };
            auto next = [&](auto Qc, int at) {
                constexpr int Q = decltype(Qc)::value;
                return V<R>{block_t<R, COMP>(s, n, Q)[at], COMP ? block_t<R, COMP>(s, n, 3 + Q)[at] : R(0)};
            };
            auto keep = [&](auto Qc, int at, V<R> v) {
                constexpr int Q = decltype(Qc)::value;
                block_t<R, COMP>(s, n, Q)[at] = v.h;
                if constexpr (COMP) block_t<R, COMP>(s, n, 3 + Q)[at] = v.l;
            };
            auto hand = [&](auto Qc, int kind, const Own<R>& g, V<R> a) {
                constexpr int Q = decltype(Qc)::value;
                if (kind != CELL_IN) return;
                keep(Qc, tid, V<R>{g.h, g.l});
                if (k == Ext<Q>::Lz(m.nz) - 1 && zp != t)
                    keep(Qc, zp, mur_map<MODE>(level(Qc, t), m.mur[9 + Q], m.mur_lo[9 + Q], a, level(Qc, zp)));
            };
            // the Mur map of the cell from the one at `from`, kept for the next pass
            auto face = [&](auto Qc, int from, R ch, R cl, V<R>& a) {
                a = mur_map<MODE>(level(Qc, from), ch, cl, next(Qc, from), level(Qc, t));
                keep(Qc, tid, a);
            };
            const std::integral_constant<int, 0> Q0;
            const std::integral_constant<int, 1> Q1;
            const std::integral_constant<int, 2> Q2;
            if (active) {
                hand(Q0, kind0, g0, a0);
                hand(Q1, kind1, g1, a1);
                hand(Q2, kind2, g2, a2);
            }
            __syncthreads();
            if (i1 >= m.nx - 1) {
                if (active) {
                    // an x face column's cells below z = max, y edges left to the y faces
                    if (kind0 == CELL_X) face(Q0, xm, m.mur[0], m.mur_lo[0], a0);
                    if (kind1 == CELL_X) face(Q1, xm, m.mur[1], m.mur_lo[1], a1);
                    if (kind2 == CELL_X) face(Q2, xm, m.mur[2], m.mur_lo[2], a2);
                }
                __syncthreads();
            }
            if (j0 == 0 || j1 >= m.ny - 1) {
                if (active) {
                    auto yface = [&](auto Qc, int kind, V<R>& a) {
                        constexpr int Q = decltype(Qc)::value;
                        const bool lo = kind == CELL_Y0;
                        if (lo || kind == CELL_Y1)
                            face(Qc, lo ? yp : ym, lo ? m.mur[3 + Q] : m.mur[6 + Q], lo ? m.mur_lo[3 + Q] : m.mur_lo[6 + Q],
                                 a);
                    };
                    yface(Q0, kind0, a0);
                    yface(Q1, kind1, a1);
                    yface(Q2, kind2, a2);
                }
                __syncthreads();
            }
            if (k1 >= m.nz - 1 && active) {
                auto zface = [&](auto Qc, int kind, V<R>& a) {
                    constexpr int Q = decltype(Qc)::value;
                    if (kind != CELL_Z) return;
                    if (face_column<Q>(m, i, j))
                        a = mur_map<MODE>(level(Qc, zm), m.mur[9 + Q], m.mur_lo[9 + Q], next(Qc, zm), level(Qc, t));
                    else
                        a = next(Qc, t);
                };
                zface(Q0, kind0, a0);
                zface(Q1, kind1, a1);
                zface(Q2, kind2, a2);
            }
            __syncthreads();  // the faces are done with level n
        }
        // rotate: cells that are none of a component's stay 0
        q0 = c0;
        q1 = c1;
        q2 = c2;
        c0 = kind0 == CELL_NONE ? zero : block_stored<MODE>(a0);
        c1 = kind1 == CELL_NONE ? zero : block_stored<MODE>(a1);
        c2 = kind2 == CELL_NONE ? zero : block_stored<MODE>(a2);
        // a recording step's frame (pr.ring: null when none of these steps is)
        const long long tt = tt0 + r;
        if (pr.ring && (tt + 1) % pr.every == 0) {
            const long long f = (tt + 1) / pr.every - 1;  // every recording step since step 0 took a frame
            if (own && k == 0 && kind2 != CELL_NONE) {
                const int pi = i - pr.i0, pj = j - pr.j0;
                if (pi >= 0 && pj >= 0 && pi % pr.si == 0 && pj % pr.sj == 0 && pi / pr.si < pr.ni && pj / pr.sj < pr.nj) {
                    double d = (double)c2.h;
                    if constexpr (COMP) d += (double)c2.l;
                    pr.ring[(f % pr.cap) * (long long)pr.ni * pr.nj + (pi / pr.si) * pr.nj + pj / pr.sj] = d;
                }
            }
            if (blockIdx.x == 0 && tid == 0) *pr.frame = f + 1;
        }
        if (r + 1 < steps) publish(tt + 1);
    }
    if (!own) return;
    if (kind0 != CELL_NONE) block_put<MODE>(m.n0, m.nl0, id, c0);
    if (kind1 != CELL_NONE) block_put<MODE>(m.n1, m.nl1, id, c1);
    if (kind2 != CELL_NONE) block_put<MODE>(m.n2, m.nl2, id, c2);
    if (steps > 1) {
        if (kind0 != CELL_NONE) block_put<MODE>(p0, pl0, id, q0);
        if (kind1 != CELL_NONE) block_put<MODE>(p1, pl1, id, q1);
        if (kind2 != CELL_NONE) block_put<MODE>(p2, pl2, id, q2);
    }
}

// What a launch costs (microseconds): `launch` once; for every round of
// resident blocks `round` to load and store, and per step a chain `chain`
// and `wave` for each wave a CU holds (waves_cu at most).  Fitted to launches
// of 1 to 4 steps on meshes of 210 to 140,000 nodes, within 15 % of each.
// `march`: the least a step of the tiled sweep and its face launch takes
// there, the line below which a mesh steps in blocks.  Measured, microseconds
// a step in blocks / marched (x chunks by the rule of tile_map): 31 x 21 x 6
// nodes FP64 with divisions 5.9 / 15.6, FP64 4.8 / 13.9, FP32 3.8 / 12.0,
// FP32C 5.7 / 17.8; 58 x 39 x 13 nodes 8.7 / 15.8, 6.1 / 13.9, 4.7 / 11.6,
// 8.1 / 16.7; 49 x 45 x 24 nodes 9.2 / 15.0, 7.3 / 13.4, 5.4 / 11.4, 8.8 /
// 16.4; 65 x 65 x 33 nodes 20.5 / 18.9, 15.7 / 16.2, 12.6 / 12.7, 21.7 / 18.1.
struct BlockCost {
    double launch, round, chain, wave;
    int waves_cu;
    double march;
};
constexpr long long BLOCK_MAX_CELLS = 300000;  // more is never below the line: spares the search
inline BlockCost block_cost(int mode) {
    switch (mode) {
        case MODE_FP64: return {1.5, 2.3, 1.2, 0.45, 12, 15.0};
        case MODE_FP64P: return {1.5, 2.3, 1.4, 0.25, 12, 13.5};
        case MODE_FP32: return {1.5, 2.3, 1.2, 0.14, 16, 11.0};
        default: return {1.5, 2.3, 1.6, 0.42, 12, 16.0};
    }
}

// The partition for launches of `steps` steps on a device of `cus` compute
// units: the one of the smallest expected time *us.  threads = 0 when none
// fits.
inline BlockMap block_map(int nx, int ny, int nz, int steps, int cus, const BlockCost& bc, double* us) {
    BlockMap best = {0, 0, 0, steps, 0};
    double best_t = 0;
    auto part = [&](int len, int nt) {  // nodes of the largest box along an axis
        const int w = (len + nt - 1) / nt + (nt == 1 ? 0 : nt == 2 ? 1 : 2) * steps;
        return w < len ? w : len;
    };
    for (int ntz = 1; ntz <= nz / 3; ntz++) {
        const int ez = part(nz, ntz);
        if (ez > BLOCK_MAX_NODES) continue;
        for (int nty = 1; nty <= ny / 3; nty++) {
            const int eyz = ez * part(ny, nty);
            if (eyz > BLOCK_MAX_NODES) continue;
            for (int ntx = 1; ntx <= nx / 3; ntx++) {
                const int nodes = eyz * part(nx, ntx);
                if (nodes > BLOCK_MAX_NODES) continue;
                const int waves = (nodes + 63) / 64;
                const long long per_cu = ((long long)ntx * nty * ntz + cus - 1) / cus;
                const long long fit = waves <= 8 ? bc.waves_cu / waves : 1;
                const long long held = per_cu < fit ? per_cu : fit;
                const double t = bc.launch + (double)((per_cu + held - 1) / held) *
                                                 (bc.round + steps * (bc.chain + bc.wave * (double)(held * waves)));
                if (best.threads == 0 || t < best_t * 0.9999) {
                    best = {ntx, nty, ntz, steps, waves * 64};
                    best_t = t;
                }
            }
        }
    }
    if (us) *us = best_t;
    return best;
}

template <class R, int MODE, bool SPONGE, int MOST>
int launch_block_m(const Mesh<R>& m, const BlockMap& bm, R* const* p, lo_t* const* pl, const FaceProbe& pr,
                   hipStream_t s) {
    const auto kernel = k_block_steps<R, MODE, SPONGE, MOST>;
    const size_t lds = block_lds<R, MODE>(bm.threads);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(bm.ntx * bm.nty * bm.ntz)), dim3((unsigned)bm.threads), lds, s, m, p[0],
                       p[1], p[2], pl[0], pl[1], pl[2], bm, bm.steps, pr);
    HIPCHK(hipGetLastError());
    return PF_OK;
}

// Blocks of at most 512 threads may use twice the registers (the FP64 and
// FP32C flavours spill a few within 128).
template <class R, int MODE, bool SPONGE>
int launch_block_k(const Mesh<R>& m, const BlockMap& bm, R* const* p, lo_t* const* pl, const FaceProbe& pr,
                   hipStream_t s) {
    return bm.threads <= 512 ? launch_block_m<R, MODE, SPONGE, 512>(m, bm, p, pl, pr, s)
                             : launch_block_m<R, MODE, SPONGE, BLOCK_MAX_NODES>(m, bm, p, pl, pr, s);
}

// Allows the kernel that takes blocks of bm its LDS on the current device (only
// the largest blocks in FP64 need more than every kernel may have).
template <class R, int MODE, bool SPONGE>
hipError_t allow_block_k(const BlockMap& bm) {
    const size_t lds = block_lds<R, MODE>(bm.threads);
    if (lds <= 64u << 10) return hipSuccess;
    const void* kernel = bm.threads <= 512 ? (const void*)k_block_steps<R, MODE, SPONGE, 512>
                                           : (const void*)k_block_steps<R, MODE, SPONGE, BLOCK_MAX_NODES>;
    return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)block_lds<R, MODE>(BLOCK_MAX_NODES));
}

}  // namespace pf
