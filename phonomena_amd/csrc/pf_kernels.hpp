// Device side of the FDTD step: mesh view, stress/displacement stencils, the
// naive sweep, the boundary-face kernel with the probes, pack/unpack.
//
// Layout in HBM (one mesh): each displacement component is a dense
// (nx, ny, pz) array, z contiguous, row stride pz (= nz: unpadded), for two
// time levels (ping-pong); a level's arrays lie back to back in one
// allocation.  Cells outside a component's reference extent (ux has nx-1
// planes, uy ny-1 rows, uz nz-1 columns) are allocated, never written and
// stay zero.  Material: one uint8 index per node in the same layout, and a
// 16-value row per material.
//
// Semantics of one step (what the reference does in base_solver.py:245-256):
//   1. the wall line uz[0, :, 0] takes the source value w(tt); here the value
//      is substituted on every read of that line instead of being stored;
//   2. stresses from u (T is never stored: each stencil recomputes it);
//   3. "stage I": the interior and free-surface displacement update;
//   4. the four Mur faces, x=max, y=0, y=max, z=max, each reading the plane
//      one cell inside as updated so far and overwriting shared edges;
//   5. rotation: the new level becomes current (pointer swap).
// Stage 4 is resolved per cell: the last face that writes a cell fixes its
// value as a chain  face(... face(stageI(inner cell)))  of at most four maps,
// and every stage-I value a chain reads lies strictly inside all faces, where
// the sweep kernel has already written it.  So the sweep writes all non-face
// cells plus the z = max face cells (a single map of the cell below), and a
// second, small kernel writes the other face cells.  Cells of uy/uz on the
// x = 0 wall that the reference never updates are written as 0, which is
// what the reference holds there (the source line included, whose stored
// value after a step is the never-written 0 of u_new).
#pragma once
#include "pf_formulas.hpp"

namespace pf {

template <class R>
struct Mesh {
    int nx, ny, nz, pz;
    long long plane;  // ny * pz
    // level n (current), hi part
    const R* __restrict__ c0;
    const R* __restrict__ c1;
    const R* __restrict__ c2;
    // level written by the step (level n+1), hi part
    R* n0;
    R* n1;
    R* n2;
    // level n-1 (read at the node only; the same arrays as n* when the step
    // overwrites the previous level in place)
    const R* o0;
    const R* o1;
    const R* o2;
    // lo parts (PF_FP32C only), 16-bit (lo_encode / lo_decode)
    const lo_t* __restrict__ cl0;
    const lo_t* __restrict__ cl1;
    const lo_t* __restrict__ cl2;
    lo_t* nl0;
    lo_t* nl1;
    lo_t* nl2;
    const lo_t* ol0;
    const lo_t* ol1;
    const lo_t* ol2;
    const uint8_t* __restrict__ ids;
    const R* __restrict__ mat;
    // spacing tables: FP64 = spacings, FP32 = inverse spacings
    const R* __restrict__ fx;
    const R* __restrict__ fy;
    const R* __restrict__ fz;
    const R* __restrict__ sx;
    const R* __restrict__ sy;
    const R* __restrict__ sz;
    R fx0, fy0, fz0, sx0, sy0, sz0;
    // FP64: reciprocals of the spacings (the same tables, MODE_FP64Q)
    const R* __restrict__ rfx;
    const R* __restrict__ rfy;
    const R* __restrict__ rfz;
    const R* __restrict__ rsx;
    const R* __restrict__ rsy;
    const R* __restrict__ rsz;
    R rfx0, rfy0, rfz0, rsx0, rsy0, rsz0;
    const R* __restrict__ dpx;  // sponge terms per axis (null: none)
    const R* __restrict__ dpy;
    const R* __restrict__ dpz;
    R mur[12];
    R mur_lo[12];  // FP32C: low parts of the Mur coefficients
    const double* __restrict__ wave;
    const long long* __restrict__ step_base;  // device step counter or null
    long long step_off;                       // tt = *step_base + step_off
    long long nsteps;                         // step budget (batch members)
    int nmat;                                 // rows in mat
    int surf;  // 1: the surface u_z update divides T3's difference by fdz (extension); 0: the reference's precedence
};

template <class R>
PF_DEV long long at(const Mesh<R>& m, int i, int j, int k) {
    return (long long)i * m.plane + (long long)j * m.pz + k;
}

// The spacings a sweep of MODE reads: with MODE_FP64P the tables and first
// spacings are the exact reciprocals.
template <int MODE, class R>
inline void take_spacings(Mesh<R>& m) {
    if constexpr (MODE == MODE_FP64P) {
        m.fx = m.rfx; m.fy = m.rfy; m.fz = m.rfz;
        m.sx = m.rsx; m.sy = m.rsy; m.sz = m.rsz;
        m.fx0 = m.rfx0; m.fy0 = m.rfy0; m.fz0 = m.rfz0;
        m.sx0 = m.rsx0; m.sy0 = m.rsy0; m.sz0 = m.rsz0;
    }
}

template <class R>
PF_DEV long long step_index(const Mesh<R>& m) {
    return (m.step_base ? *m.step_base : 0) + m.step_off;
}

// Component extents: last valid index per axis.
template <int Q> struct Ext;
template <> struct Ext<0> { static PF_DEV int Lx(int nx) { return nx - 2; } static PF_DEV int Ly(int ny) { return ny - 1; } static PF_DEV int Lz(int nz) { return nz - 1; } };
template <> struct Ext<1> { static PF_DEV int Lx(int nx) { return nx - 1; } static PF_DEV int Ly(int ny) { return ny - 2; } static PF_DEV int Lz(int nz) { return nz - 1; } };
template <> struct Ext<2> { static PF_DEV int Lx(int nx) { return nx - 1; } static PF_DEV int Ly(int ny) { return ny - 1; } static PF_DEV int Lz(int nz) { return nz - 2; } };

// ---------------------------------------------------------------- loads ----
template <class R> PF_DEV R lux(const Mesh<R>& m, int i, int j, int k) { return m.c0[at(m, i, j, k)]; }
template <class R> PF_DEV R luy(const Mesh<R>& m, int i, int j, int k) { return m.c1[at(m, i, j, k)]; }
template <class R> PF_DEV R luz(const Mesh<R>& m, int i, int j, int k, R w) {
    R v = m.c2[at(m, i, j, k)];
    return (i == 0 && k == 0) ? w : v;
}
template <class R> PF_DEV const R* matp(const Mesh<R>& m, int i, int j, int k) {
    return m.mat + MAT_STRIDE * (int)m.ids[at(m, i, j, k)];
}

// ------------------------------------------------------------- stresses ----
// Each returns the value the reference's T array holds at (i,j,k) after
// update_T + apply_T_tfbc, and 0 where the reference never writes it.
template <int EXACT, class R>
PF_DEV void tn(const Mesh<R>& m, int i, int j, int k, R w, R& t1, R& t2, R& t3) {
    t1 = t2 = t3 = R(0);
    if (i < 1 || i > m.nx - 2 || j < 1 || j > m.ny - 2 || k < 0 || k > m.nz - 2) return;
    const R* c = matp(m, i, j, k);
    R dux = lux(m, i, j, k) - lux(m, i - 1, j, k);
    R duy = luy(m, i, j, k) - luy(m, i, j - 1, k);
    if (k >= 1) {
        R duz = luz(m, i, j, k, w) - luz(m, i, j, k - 1, w);
        normal3<EXACT>(c, dux, duy, duz, m.sx[i - 1], m.sy[j - 1], m.sz[k - 1], t1, t2, t3);
    } else {
        normal3_surface<EXACT>(c, dux, duy, luz(m, i, j, 0, w), m.sx0, m.sy0, m.sz0, t1, t2, t3);
    }
}

template <int EXACT, class R>
PF_DEV R t4(const Mesh<R>& m, int i, int j, int k, R w) {
    if (i < 1 || i > m.nx - 2 || j < 0 || j > m.ny - 2 || k < 0 || k > m.nz - 2) return R(0);
    if (k >= 1) {
        R c = matp(m, i, j + 1, k + 1)[M_C33];
        return shear<EXACT>(c, luy(m, i, j, k + 1) - luy(m, i, j, k), m.fz[k],
                            luz(m, i, j + 1, k, w) - luz(m, i, j, k, w), m.fy[j]);
    }
    R c = matp(m, i, j + 1, 0)[M_C33];
    return shear<EXACT>(c, luy(m, i, j, 1) - luy(m, i, j, 0), m.fy0,
                        luz(m, i, j + 1, 0, w) - luz(m, i, j, 0, w), m.fz0);
}

template <int EXACT, class R>
PF_DEV R t5(const Mesh<R>& m, int i, int j, int k, R w) {
    if (i < 0 || i > m.nx - 2 || j < 1 || j > m.ny - 2 || k < 0 || k > m.nz - 2) return R(0);
    if (k >= 1) {
        R c = matp(m, i + 1, j, k + 1)[M_C44];
        return shear<EXACT>(c, lux(m, i, j, k + 1) - lux(m, i, j, k), m.fz[k],
                            luz(m, i + 1, j, k, w) - luz(m, i, j, k, w), m.fx[i]);
    }
    R c = matp(m, i + 1, j, 0)[M_C44];
    return shear<EXACT>(c, lux(m, i, j, 1) - lux(m, i, j, 0), m.fx0,
                        luz(m, i + 1, j, 0, w) - luz(m, i, j, 0, w), m.fz0);
}

template <int EXACT, class R>
PF_DEV R t6(const Mesh<R>& m, int i, int j, int k, R w) {
    if (i < 0 || i > m.nx - 2 || j < 0 || j > m.ny - 2 || k < 0 || k > m.nz - 2) return R(0);
    (void)w;
    if (k >= 1) {
        R c = matp(m, i + 1, j + 1, k)[M_C55];
        return shear<EXACT>(c, lux(m, i, j + 1, k) - lux(m, i, j, k), m.fy[j],
                            luy(m, i + 1, j, k) - luy(m, i, j, k), m.fx[i]);
    }
    R c = matp(m, i + 1, j + 1, 0)[M_C55];
    return shear<EXACT>(c, lux(m, i, j + 1, 0) - lux(m, i, j, 0), m.fx0,
                        luy(m, i + 1, j, 0) - luy(m, i, j, 0), m.fz0);
}

template <class R>
PF_DEV R damp_at(const Mesh<R>& m, int i, int j, int k) {
    return m.dpx[i] + m.dpy[j] + m.dpz[k];
}

// Stage-I bracket ("div") and coefficient of each component at a non-face
// cell (base_solver.py:441-463 for k >= 1, :495-517 for k = 0).
template <int EXACT, class R>
PF_DEV void stage_ux(const Mesh<R>& m, int i, int j, int k, R w, R& coef, R& dv) {
    R a1, a2, a3, b1, b2, b3;
    tn<EXACT>(m, i + 1, j, k, w, a1, a2, a3);
    tn<EXACT>(m, i, j, k, w, b1, b2, b3);
    R d6 = t6<EXACT>(m, i, j, k, w) - t6<EXACT>(m, i, j - 1, k, w);
    if (k >= 1) {
        R d5 = t5<EXACT>(m, i, j, k, w) - t5<EXACT>(m, i, j, k - 1, w);
        dv = div3<EXACT>(a1 - b1, m.fx[i], d6, m.sy[j - 1], d5, m.sz[k - 1]);
        coef = matp(m, i + 1, j, k)[M_COEF];
    } else {
        R d5 = t5<EXACT>(m, i, j, 0, w) - R(0);
        dv = div3<EXACT>(a1 - b1, m.fx0, d6, m.sy0, d5, m.sz0);
        coef = matp(m, i + 1, j, 0)[M_COEF];
    }
}

template <int EXACT, class R>
PF_DEV void stage_uy(const Mesh<R>& m, int i, int j, int k, R w, R& coef, R& dv) {
    R d6 = t6<EXACT>(m, i, j, k, w) - t6<EXACT>(m, i - 1, j, k, w);
    R a1, a2, a3, b1, b2, b3;
    tn<EXACT>(m, i, j + 1, k, w, a1, a2, a3);
    tn<EXACT>(m, i, j, k, w, b1, b2, b3);
    if (k >= 1) {
        R d4 = t4<EXACT>(m, i, j, k, w) - t4<EXACT>(m, i, j, k - 1, w);
        dv = div3<EXACT>(d6, m.sx[i - 1], a2 - b2, m.fy[j], d4, m.sz[k - 1]);
        coef = matp(m, i, j + 1, k)[M_COEF];
    } else {
        R d4 = t4<EXACT>(m, i, j, 0, w) - R(0);
        dv = div3<EXACT>(d6, m.sx0, a2 - b2, m.fy0, d4, m.sz0);
        coef = matp(m, i, j + 1, 0)[M_COEF];
    }
}

template <int EXACT, class R>
PF_DEV void stage_uz(const Mesh<R>& m, int i, int j, int k, R w, R& coef, R& dv) {
    R d5 = t5<EXACT>(m, i, j, k, w) - t5<EXACT>(m, i - 1, j, k, w);
    R d4 = t4<EXACT>(m, i, j, k, w) - t4<EXACT>(m, i, j - 1, k, w);
    R a1, a2, a3, b1, b2, b3;
    tn<EXACT>(m, i, j, k + 1, w, a1, a2, a3);
    tn<EXACT>(m, i, j, k, w, b1, b2, b3);
    if (k >= 1) {
        dv = div3<EXACT>(d5, m.sx[i - 1], d4, m.sy[j - 1], a3 - b3, m.fz[k]);
        coef = matp(m, i, j, k + 1)[M_COEF];
    } else {
        dv = m.surf ? div3<EXACT>(d5, m.sx0, d4, m.sy0, a3 - b3, m.fz0)
                    : div3_uz_surface<EXACT>(d5, m.sx0, d4, m.sy0, a3, b3, m.fz0);
        coef = matp(m, i, j, 0)[M_COEF];  // reference samples rho at k = 0 here
    }
}

// ----------------------------------------------------------- faces ----
// A value in flight through the face chain: hi (+ lo in compensated mode).
template <class R> struct V { R h, l; };

template <int Q, class R>
PF_DEV V<R> cur_q(const Mesh<R>& m, int i, int j, int k, R w) {
    long long id = at(m, i, j, k);
    const R* c = Q == 0 ? m.c0 : (Q == 1 ? m.c1 : m.c2);
    const lo_t* cl = Q == 0 ? m.cl0 : (Q == 1 ? m.cl1 : m.cl2);
    V<R> v;
    v.h = c[id];
    v.l = cl ? lo_decode(v.h, cl[id]) : R(0);
    if (Q == 2 && i == 0 && k == 0) { v.h = w; v.l = R(0); }
    return v;
}

// a + c * (b - d), the reference's `q[..] + c*(q_new[..] - q[..])`
template <int MODE, class R>
PF_DEV V<R> mur_map(V<R> a, R ch, R cl, V<R> b, V<R> d) {
    V<R> r;
    if constexpr (MODE == MODE_FP32C) {
        mur_comp(a.h, a.l, ch, cl, b.h, b.l, d.h, d.l, r.h, r.l);
    } else {
        r.h = a.h + ch * (b.h - d.h);
        r.l = R(0);
    }
    return r;
}

template <int Q, class R> PF_DEV R* nptr(const Mesh<R>& m) { return Q == 0 ? m.n0 : (Q == 1 ? m.n1 : m.n2); }
template <int Q, class R> PF_DEV lo_t* nlptr(const Mesh<R>& m) { return Q == 0 ? m.nl0 : (Q == 1 ? m.nl1 : m.nl2); }

template <int Q, int MODE, class R>
PF_DEV void put(const Mesh<R>& m, int i, int j, int k, V<R> v) {
    const long long id = at(m, i, j, k);
    nptr<Q>(m)[id] = v.h;
    if constexpr (MODE == MODE_FP32C) nlptr<Q>(m)[id] = lo_encode(v.h, v.l);
}

// Write the stage-I value s0 of a non-face cell, and, when k = Lz-1, the
// z = max face cell above it, whose final value is a single Mur map of s0
// (there the data is already in the sweep's registers; a separate pass
// would read it back with a stride of one row per cell).  `cur` is the
// cell's own level-n value.
template <int Q, int MODE, class R>
PF_DEV void put_with_zface(const Mesh<R>& m, int i, int j, int k, V<R> s0, V<R> cur, R w) {
    put<Q, MODE>(m, i, j, k, s0);
    const int Lz = Ext<Q>::Lz(m.nz);
    if (k == Lz - 1)
        put<Q, MODE>(m, i, j, Lz, mur_map<MODE>(cur, m.mur[9 + Q], m.mur_lo[9 + Q], s0, cur_q<Q>(m, i, j, Lz, w)));
}

// Face cells of component Q not written by the sweep, once each, z fastest
// so each run of threads touches contiguous memory:
//   X  : (Lx, j, k)   0 < j < Ly, k < Lz
//   Y0 : (i, 0, k)    i < Lx,     k < Lz
//   Y1 : (i, Ly, k)   i < Lx,     k < Lz
//   box edges (two or more faces meet):
//        (Lx, 0, k), (Lx, Ly, k)   all k
//        (Lx, j, Lz)               0 < j < Ly
//        (i, 0, Lz), (i, Ly, Lz)   i < Lx
template <int Q>
PF_DEV int face_edges(int nx, int ny, int nz) {
    return 2 * (Ext<Q>::Lz(nz) + 1) + Ext<Q>::Ly(ny) - 1 + 2 * Ext<Q>::Lx(nx);
}

// Box-edge cell t of component Q.
template <int Q>
PF_DEV void face_edge_cell(int nx, int ny, int nz, int t, int& i, int& j, int& k) {
    const int Lx = Ext<Q>::Lx(nx), Ly = Ext<Q>::Ly(ny), Lz = Ext<Q>::Lz(nz);
    if (t < Lz + 1) { i = Lx; j = 0; k = t; return; }
    t -= Lz + 1;
    if (t < Lz + 1) { i = Lx; j = Ly; k = t; return; }
    t -= Lz + 1;
    if (t < Ly - 1) { i = Lx; j = 1 + t; k = Lz; return; }
    t -= Ly - 1;
    if (t < Lx) { i = t; j = 0; k = Lz; return; }
    i = t - Lx; j = Ly; k = Lz;
}

// Final value of a face cell: the interior cell's new value through the Mur
// maps of the faces it lies on, in the reference's order x = max, y = 0 or
// y = max, z = max (base_solver.py:525-554), each
//   face = cur(inside) + c (new(inside) - cur(face)),
// where inside is the cell one step off that face.  Each map's operands are the
// level-n values on the way from the interior cell (ii, ji, ki) to the face
// cell, so five values give all three maps, and their loads leave together
// (needs Lx >= 1, Ly >= 2, Lz >= 1, so that no step off a face ends on
// another: meshes have at least four nodes per axis).  As a recursion over the
// faces the lanes of a wave at different edges took its branches, and their
// loads, one after another.
template <int Q, int MODE, class R>
PF_DEV V<R> face_value(const Mesh<R>& m, int i, int j, int k, R w) {
    const int Lx = Ext<Q>::Lx(m.nx), Ly = Ext<Q>::Ly(m.ny), Lz = Ext<Q>::Lz(m.nz);
    const bool fx = i == Lx, fy = j == 0 || j == Ly, fz = k == Lz;
    const int ii = fx ? Lx - 1 : i, ji = j == 0 ? 1 : (j == Ly ? Ly - 1 : j), ki = fz ? Lz - 1 : k;
    const R yh = j == 0 ? m.mur[3 + Q] : m.mur[6 + Q], yl = j == 0 ? m.mur_lo[3 + Q] : m.mur_lo[6 + Q];
    const R* cp = Q == 0 ? m.c0 : (Q == 1 ? m.c1 : m.c2);
    const R* np = nptr<Q>(m);
    const long long ia = at(m, ii, ji, ki), ib = at(m, i, ji, ki), ic = at(m, i, j, ki), id = at(m, i, j, k);
    V<R> v = {np[ia], R(0)}, a = {cp[ia], R(0)}, b = {cp[ib], R(0)}, c = {cp[ic], R(0)}, d = {cp[id], R(0)};
    if constexpr (MODE == MODE_FP32C) {
        const lo_t* cl = Q == 0 ? m.cl0 : (Q == 1 ? m.cl1 : m.cl2);
        const lo_t lv = nlptr<Q>(m)[ia], la = cl[ia], lb = cl[ib], lc = cl[ic], ld = cl[id];
        v.l = lo_decode(v.h, lv);
        a.l = lo_decode(a.h, la);
        b.l = lo_decode(b.h, lb);
        c.l = lo_decode(c.h, lc);
        d.l = lo_decode(d.h, ld);
    }
    if (Q == 2) {  // the source line uz[0, :, 0] reads as w
        const V<R> src = {w, R(0)};
        if (ii == 0 && ki == 0) a = src;
        if (i == 0 && ki == 0) b = c = src;
        if (i == 0 && k == 0) d = src;
    }
    const V<R> x = mur_map<MODE>(a, m.mur[0 + Q], m.mur_lo[0 + Q], v, b);
    v = {fx ? x.h : v.h, fx ? x.l : v.l};
    const V<R> y = mur_map<MODE>(b, yh, yl, v, c);
    v = {fy ? y.h : v.h, fy ? y.l : v.l};
    const V<R> z = mur_map<MODE>(c, m.mur[9 + Q], m.mur_lo[9 + Q], v, d);
    return {fz ? z.h : v.h, fz ? z.l : v.l};
}

// The rows of the three face planes
//   X  (Lx, j, k)  0 < j < Ly,   Y0 (i, 0, k), Y1 (i, Ly, k)  i < Lx,   k < Lz
// take one Mur map of interior cells each:
//   X  map(cur(Lx-1, j, k), new(Lx-1, j, k), cur(Lx, j, k))
//   Y0 map(cur(i, 1, k),    new(i, 1, k),    cur(i, 0, k))
//   Y1 map(cur(i, Ly-1, k), new(i, Ly-1, k), cur(i, Ly, k))
// (face_value with the one face).  The rows are cut into
// segments of 64 cells; a wave takes FACE_WAVE_SEGS of them, of as many rows as
// that is, and issues all its loads before it stores anything, so one round of
// memory latency covers them.  The launch is bound by that round and its fixed
// cost, about 4 us (513 x 513 x 257 nodes FP32 7.2 us, 257 x 257 x 129 FP32C
// 5.4; two segments a wave 8.1 and 5.6, eight 7.6 and 6.4; with rows of up to
// 256 cells a wave and the edges one a thread through a recursion 8.4 and
// 9.1).  The box edges, a few thousand cells, go to blocks of their own, the
// last ones (measured 0.4 us faster per launch than putting them first).
constexpr int FACE_WAVE_SEGS = 4;
PF_DEV int face_segs(int nz) { return (nz - 1 + 63) / 64; }

template <int Q>
PF_DEV int face_rows(int nx, int ny) {
    return Ext<Q>::Ly(ny) - 1 + 2 * Ext<Q>::Lx(nx);
}
// Waves of component Q's rows.
template <int Q>
PF_DEV int face_waves(int nx, int ny, int nz) {
    return (face_rows<Q>(nx, ny) * face_segs(nz) + FACE_WAVE_SEGS - 1) / FACE_WAVE_SEGS;
}

// Wave t of component Q's rows.
template <int Q, int MODE, class R>
PF_DEV void face_row_wave(const Mesh<R>& m, int t, int lane, R w) {
    const int Lx = Ext<Q>::Lx(m.nx), Ly = Ext<Q>::Ly(m.ny), Lz = Ext<Q>::Lz(m.nz);
    const int ks = face_segs(m.nz), last = face_rows<Q>(m.nx, m.ny) * ks - 1;
    const R* c = Q == 0 ? m.c0 : (Q == 1 ? m.c1 : m.c2);
    const R* n = Q == 0 ? m.n0 : (Q == 1 ? m.n1 : m.n2);
    const lo_t* cl = Q == 0 ? m.cl0 : (Q == 1 ? m.cl1 : m.cl2);
    const lo_t* nl = Q == 0 ? m.nl0 : (Q == 1 ? m.nl1 : m.nl2);
    V<R> a[FACE_WAVE_SEGS], b[FACE_WAVE_SEGS], d[FACE_WAVE_SEGS];
    int i[FACE_WAVE_SEGS], j[FACE_WAVE_SEGS], ii[FACE_WAVE_SEGS], k[FACE_WAVE_SEGS];
    R mh[FACE_WAVE_SEGS], ml[FACE_WAVE_SEGS];
#pragma unroll
    for (int u = 0; u < FACE_WAVE_SEGS; u++) {
        // the face row, the interior row its map reads, its Mur coefficient
        // (constant indices: a run-time index into the kernel argument would
        // copy it to scratch)
        const int g = t * FACE_WAVE_SEGS + u < last ? t * FACE_WAVE_SEGS + u : last;
        const int r = g / ks;
        int ji;
        if (r < Ly - 1) {
            i[u] = Lx; j[u] = 1 + r; ii[u] = Lx - 1; ji = j[u]; mh[u] = m.mur[0 + Q]; ml[u] = m.mur_lo[0 + Q];
        } else if (r < Ly - 1 + Lx) {
            i[u] = r - (Ly - 1); j[u] = 0; ii[u] = i[u]; ji = 1; mh[u] = m.mur[3 + Q]; ml[u] = m.mur_lo[3 + Q];
        } else {
            i[u] = r - (Ly - 1) - Lx; j[u] = Ly; ii[u] = i[u]; ji = Ly - 1; mh[u] = m.mur[6 + Q]; ml[u] = m.mur_lo[6 + Q];
        }
        const long long fb = at(m, i[u], j[u], 0), ib = at(m, ii[u], ji, 0);
        k[u] = (g - r * ks) * 64 + lane;
        const int kk = k[u] < Lz ? k[u] : Lz - 1;  // lanes past the row load its last cell and store nothing
        if (t * FACE_WAVE_SEGS + u > last) k[u] = Lz;
        a[u].h = c[ib + kk];
        b[u].h = n[ib + kk];
        d[u].h = c[fb + kk];
        if constexpr (MODE == MODE_FP32C) {
            a[u].l = lo_decode(a[u].h, cl[ib + kk]);
            b[u].l = lo_decode(b[u].h, nl[ib + kk]);
            d[u].l = lo_decode(d[u].h, cl[fb + kk]);
        } else {
            a[u].l = b[u].l = d[u].l = R(0);
        }
    }
#pragma unroll
    for (int u = 0; u < FACE_WAVE_SEGS; u++) {
        if (k[u] >= Lz) continue;
        if (Q == 2 && k[u] == 0) {  // the source line uz[0, :, 0] reads as w
            if (ii[u] == 0) { a[u].h = w; a[u].l = R(0); }
            if (i[u] == 0) { d[u].h = w; d[u].l = R(0); }
        }
        put<Q, MODE>(m, i[u], j[u], k[u], mur_map<MODE>(a[u], mh[u], ml[u], b[u], d[u]));
    }
}

// The faces read no spacings: one kernel serves all FP64 modes.
constexpr int face_mode(int mode) { return mode == MODE_FP64P || mode == MODE_FP64Q ? MODE_FP64 : mode; }

// A probe frame recorded by the face launch (probe blocks after the row
// and edge blocks; blocks = 0: none).
struct FaceProbe {
    double* ring;
    long long* frame;
    int* done;
    int i0, si, ni, j0, sj, nj, cap, every, blocks;
};

// Probe point p of the u_z surface (k = 0) of the level m writes, as a later
// read would see it.  Points on a u_z face (i = Lx, j = 0 or Ly) are not
// read: the face blocks of the same launch store them, so the point takes
// the same value (face_value) with its lo part rounded as stored.
template <class R, int MODE>
PF_DEV double probe_point(const Mesh<R>& m, const FaceProbe& pr, int p, R w) {
    const int i = pr.i0 + pr.si * (p / pr.nj), j = pr.j0 + pr.sj * (p % pr.nj);
    if (i == Ext<2>::Lx(m.nx) || j == 0 || j == Ext<2>::Ly(m.ny)) {
        const V<R> v = face_value<2, MODE>(m, i, j, 0, w);
        double d = (double)v.h;
        if constexpr (MODE == MODE_FP32C) d += (double)lo_decode(v.h, lo_encode(v.h, v.l));
        return d;
    }
    const long long id = at(m, i, j, 0);
    const R h = m.n2[id];
    double d = (double)h;
    if (m.nl2) d += (double)lo_decode(h, m.nl2[id]);
    return d;
}

// Row block rb of k_faces_rows' grid (four waves) for the view that view()
// gives, asked once the component is known: a batch's view is loaded from
// memory, and only what the component needs of it should be.
template <class R, int MODE, class View>
PF_DEV void face_rows_block(int nx, int ny, int nz, const View& view, int rb, R w) {
    const int lane = threadIdx.x % 64;
    int t = __builtin_amdgcn_readfirstlane(rb * 4 + (int)threadIdx.x / 64);  // this wave
    const int w0 = face_waves<0>(nx, ny, nz);
    if (t < w0) { face_row_wave<0, MODE, R>(view(), t, lane, w); return; }
    t -= w0;
    const int w1 = face_waves<1>(nx, ny, nz);
    if (t < w1) { face_row_wave<1, MODE, R>(view(), t, lane, w); return; }
    t -= w1;
    if (t < face_waves<2>(nx, ny, nz)) face_row_wave<2, MODE, R>(view(), t, lane, w);
}

// Box-edge cell e of component Q.
template <int Q, int MODE, class R>
PF_DEV void face_edge(const Mesh<R>& m, int e, R w) {
    int i, j, k;
    face_edge_cell<Q>(m.nx, m.ny, m.nz, e, i, j, k);
    put<Q, MODE>(m, i, j, k, face_value<Q, MODE>(m, i, j, k, w));
}

// Edge block eb for view m: FACE_EDGES box-edge cells, spread over its waves.
// Most edges run along x or y, so each cell reads ten cache lines of its own,
// and a CU has only so many misses in flight: few cells a block.
constexpr int FACE_EDGES = 64;
template <class R, int MODE>
PF_DEV void face_edges_block(const Mesh<R>& m, int eb, R w) {
    constexpr int PER = FACE_EDGES / 4;  // a wave's cells
    const int lane = threadIdx.x % 64;
    if (lane >= PER) return;
    int e = eb * FACE_EDGES + (int)threadIdx.x / 64 * PER + lane;
    const int e0 = face_edges<0>(m.nx, m.ny, m.nz);
    if (e < e0) { face_edge<0, MODE>(m, e, w); return; }
    e -= e0;
    const int e1 = face_edges<1>(m.nx, m.ny, m.nz);
    if (e < e1) { face_edge<1, MODE>(m, e, w); return; }
    e -= e1;
    if (e < face_edges<2>(m.nx, m.ny, m.nz)) face_edge<2, MODE>(m, e, w);
}

template <class R, int MODE>
__global__ __launch_bounds__(256) void k_faces_rows(Mesh<R> m, int row_blocks, int edge_blocks, FaceProbe pr) {
    __shared__ int s_last;
    const long long tt = step_index(m);
    if (tt >= m.nsteps) return;
    const R w = (R)m.wave[tt];
    if ((int)blockIdx.x >= row_blocks + edge_blocks) {
        // probe blocks: the frame of a recording step (the same for every block)
        if ((tt + 1) % pr.every != 0) return;
        const long long f = *pr.frame;
        const int p = ((int)blockIdx.x - row_blocks - edge_blocks) * 256 + (int)threadIdx.x;
        if (p < pr.ni * pr.nj) pr.ring[(f % pr.cap) * (long long)pr.ni * pr.nj + p] = probe_point<R, MODE>(m, pr, p, w);
        __syncthreads();
        if (threadIdx.x == 0) {
            __threadfence();
            s_last = atomicAdd(pr.done, 1) == pr.blocks - 1;
        }
        __syncthreads();
        if (s_last && threadIdx.x == 0) {
            *pr.frame = f + 1;
            *pr.done = 0;
        }
        return;
    }
    if ((int)blockIdx.x < row_blocks)
        face_rows_block<R, MODE>(m.nx, m.ny, m.nz, [&]() -> const Mesh<R>& { return m; }, (int)blockIdx.x, w);
    else face_edges_block<R, MODE>(m, (int)blockIdx.x - row_blocks, w);
}

// Blocks of k_faces_rows for an nx x ny x nz mesh: row_blocks (four waves
// each), then edge_blocks.
inline void face_rows_grid(int nx, int ny, int nz, long long& row_blocks, long long& edge_blocks) {
    const long long ks = (nz - 1 + 63) / 64;
    long long waves = 0, edges = 0;
    const long long L[3][3] = {{nx - 2, ny - 1, nz - 1}, {nx - 1, ny - 2, nz - 1}, {nx - 1, ny - 1, nz - 2}};
    for (const auto& e : L) {
        waves += ((e[1] - 1 + 2 * e[0]) * ks + FACE_WAVE_SEGS - 1) / FACE_WAVE_SEGS;
        edges += 2 * (e[2] + 1) + (e[1] - 1) + 2 * e[0];
    }
    row_blocks = (waves + 3) / 4;
    edge_blocks = (edges + FACE_EDGES - 1) / FACE_EDGES;
}

// Stage-I value of one component at a cell: the leapfrog of its current
// value cur (hi + lo), its previous value (oh + ol) and coef*div.
template <int MODE, bool SPONGE, class R>
PF_DEV V<R> leap_from(V<R> cur, R oh, R ol, R coef, R dv, R s) {
    V<R> r;
    if constexpr (MODE == MODE_FP32C) {
        leap_comp<SPONGE>(cur.h, cur.l, oh, ol, coef * dv, s, r.h, r.l);
    } else {
        r.h = leap<exact_of(MODE), SPONGE>(cur.h, oh, coef, dv, s);
        r.l = R(0);
    }
    return r;
}

template <int MODE, bool SPONGE, class R>
PF_DEV V<R> leap_value(V<R> cur, const R* nh, const lo_t* nl, long long id, R coef, R dv, R s) {
    const R oh = nh[id];
    return leap_from<MODE, SPONGE>(cur, oh, nl ? lo_decode(oh, nl[id]) : R(0), coef, dv, s);
}

// ------------------------------------------------------- naive sweep ----
// One node (i, j, k) of a step: every stress a stencil needs is recomputed
// from u.  Writes the node's non-face cells and the z = max face cells
// above them.
template <class R, int MODE, bool SPONGE>
PF_DEV void naive_cell(const Mesh<R>& m, int i, int j, int k, R w) {
    constexpr int EXACT = exact_of(MODE);
    const long long id = at(m, i, j, k);
    const R s = SPONGE ? damp_at(m, i, j, k) : R(0);
    // ux: non-face cells i <= nx-3, 1 <= j <= ny-2, k <= nz-2
    if (i <= m.nx - 3 && j >= 1 && j <= m.ny - 2 && k <= m.nz - 2) {
        R coef, dv;
        stage_ux<EXACT>(m, i, j, k, w, coef, dv);
        V<R> cur = cur_q<0>(m, i, j, k, w);
        put_with_zface<0, MODE>(m, i, j, k, leap_value<MODE, SPONGE>(cur, m.o0, m.ol0, id, coef, dv, s), cur, w);
    }
    // uy: non-face cells i <= nx-2, 1 <= j <= ny-3, k <= nz-2; wall i = 0 -> 0
    if (i <= m.nx - 2 && j >= 1 && j <= m.ny - 3 && k <= m.nz - 2) {
        V<R> cur = cur_q<1>(m, i, j, k, w);
        V<R> s0 = {R(0), R(0)};
        if (i > 0) {
            R coef, dv;
            stage_uy<EXACT>(m, i, j, k, w, coef, dv);
            s0 = leap_value<MODE, SPONGE>(cur, m.o1, m.ol1, id, coef, dv, s);
        }
        put_with_zface<1, MODE>(m, i, j, k, s0, cur, w);
    }
    // uz: non-face cells i <= nx-2, 1 <= j <= ny-2, k <= nz-3; wall i = 0 -> 0
    if (i <= m.nx - 2 && j >= 1 && j <= m.ny - 2 && k <= m.nz - 3) {
        V<R> cur = cur_q<2>(m, i, j, k, w);
        V<R> s0 = {R(0), R(0)};
        if (i > 0) {
            R coef, dv;
            stage_uz<EXACT>(m, i, j, k, w, coef, dv);
            s0 = leap_value<MODE, SPONGE>(cur, m.o2, m.ol2, id, coef, dv, s);
        }
        put_with_zface<2, MODE>(m, i, j, k, s0, cur, w);
    }
}

// One thread per node.
template <class R, int MODE, bool SPONGE>
__global__ __launch_bounds__(256) void k_sweep_naive(Mesh<R> m) {
    const int k = blockIdx.x * 64 + threadIdx.x;
    const int j = blockIdx.y * 4 + threadIdx.y;
    const int i = blockIdx.z;
    if (k >= m.nz || j >= m.ny || i >= m.nx) return;
    const long long tt = step_index(m);
    if (tt >= m.nsteps) return;
    naive_cell<R, MODE, SPONGE>(m, i, j, k, (R)m.wave[tt]);
}

// ------------------------------------------------------- pack/unpack ----
// Dense reference-shaped double array <-> padded device component: elements
// first .. first + count - 1 of the array, at out[0 ..] / from in[0 ..].
template <class R>
__global__ void k_pack(const R* __restrict__ hi, const lo_t* __restrict__ lo, long long plane, int pz,
                       int ey, int ez, long long first, long long count, double* __restrict__ out,
                       const double* __restrict__ wsub) {
    const long long o = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= count) return;
    const long long t = first + o;
    int k = (int)(t % ez);
    long long r = t / ez;
    int j = (int)(r % ey);
    int i = (int)(r / ey);
    long long id = (long long)i * plane + (long long)j * pz + k;
    const R h = hi[id];
    double v = (double)h;
    if (lo) v += (double)lo_decode(h, lo[id]);
    if (wsub && i == 0 && k == 0) v = *wsub;  // the source value on the wall line
    out[o] = v;
}

template <class R>
__global__ void k_unpack(R* __restrict__ hi, lo_t* __restrict__ lo, long long plane, int pz,
                         int ey, int ez, long long first, long long count, const double* __restrict__ in) {
    const long long o = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= count) return;
    const long long t = first + o;
    int k = (int)(t % ez);
    long long r = t / ez;
    int j = (int)(r % ey);
    int i = (int)(r / ey);
    long long id = (long long)i * plane + (long long)j * pz + k;
    double v = in[o];
    R h = (R)v;
    hi[id] = h;
    if (lo) lo[id] = lo_encode(h, (R)(v - (double)h));
}

}  // namespace pf
