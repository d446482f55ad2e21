// lee_rk_row.h -- an RK4 stage in row form (lee_row.h): one launch over the air, the porous
// layer, every face and the receivers (two over a large grid, whose interior outside every
// layer runs a kernel without layer terms), or over all members of an ensemble.
//
// The general form takes three launches a stage and, for a layer point, reads and writes the
// stage state and the accumulator of four auxiliaries per slab in every stage (68 words per slab
// element and step).  Here the auxiliaries' stage values are formed from Q_n and the previous
// stage's fields (RkRowArgs) and written once a step: 20 words, and no slab is written in three
// of the four stages.  Faces as in lee_fb.hip.
//
// Bound by memory in the interior and by the latency of its loads where layers overlap (one to
// three waves per SIMD).  Per step, MI355X, general form -> row form: 137 x 91 x 53 FP64 over
// terrain with wind and a porous layer 362 -> 267 us, 512 x 256 x 128 FP32 2224 -> 1779 us and
// FP64 3872 -> 3480 us, 768 x 384 x 192 FP32 5740 -> 4840 us, an ensemble of 32 uneven members
// up to 128 x 96 x 64 FP32 2290 -> 1810 us.  Tried and left out: three FP64 waves per SIMD
// (100-190 B of scratch a lane, 0.80-0.83x) and planes padded to a multiple of the 8 XCDs
// (0.97-1.006x).
//
// Instantiated per precision in lee_rk32.hip and lee_rk64.hip (ST: 0 first, 1 the two middle
// stages, 3 last; the register update is the stage's at compile time).
#include "lee_row.h"

#include <algorithm>

namespace lee {

namespace {

enum { RK_AIR = 0, RK_PORE = 1, RK_REC = 3 };

// Classical RK4 weights b_s and steps a_s; ca is a_s (0.5 in stages 0 and 1, 1 in stage 2).
template <typename T, int ST> constexpr T rk_w() { return (ST == 0 || ST == 3) ? T(1.0 / 6.0) : T(1.0 / 3.0); }

// The register update of a point's field: destination from level n (xn), the increment k and
// the accumulator.  FP64: acc sums x_n + sum b_s k_s.  FP32 (COMP): acc sums the increments
// alone and the last stage adds them to x_n with an exact TwoSum whose rounding error is
// carried into the next step.
template <typename T, int ST>
__device__ __forceinline__ T rk_point(T xn, T k, T acc, T err, T ca, T &acc_out, T &err_out)
{
    constexpr bool COMP = std::is_same<T, float>::value;
    constexpr T w = rk_w<T, ST>();
    if constexpr (!COMP) {
        if constexpr (ST == 0) { acc_out = xn + w * k; return xn + ca * k; }
        if constexpr (ST == 1) { acc_out = acc + w * k; return xn + ca * k; }
        return acc + w * k;
    } else {
        if constexpr (ST == 0) { acc_out = w * k; return xn + ca * k; }
        if constexpr (ST == 1) { acc_out = acc + w * k; return xn + ca * k; }
        const T y = (acc + w * k) + err;
        const T x = xn + y;
        const T bb = x - xn;
        err_out = (xn - (x - bb)) + (y - bb);  // TwoSum: xn + y = x + err exactly
        return x;
    }
}

// Lawson (integrating-factor) RK4 of a porous velocity, as rk_update_if (lee_kernels.hip) on
// values; cf = {E, E2, E2/2, E/6, E2/3}, st the stage.
template <typename T, int ST>
__device__ __forceinline__ T rk_point_if(int st, T xn, T k, T acc, T lo, T err, const T (&cf)[5], T &acc_out, T &lo_out, T &err_out)
{
    constexpr bool COMP = std::is_same<T, float>::value;
    const T E = cf[0], E2 = cf[1];
    const T w = ST == 0 ? cf[3] : ST == 1 ? cf[4] : T(1.0 / 6.0);
    const T cn = st == 2 ? E : E2, an = ST == 0 ? cf[2] : st == 1 ? T(0.5) : E2;
    if constexpr (!COMP) {
        if constexpr (ST == 0) { acc_out = E * xn + w * k; return cn * xn + an * k; }
        if constexpr (ST == 1) { acc_out = acc + w * k; return cn * xn + an * k; }
        return acc + w * k;
    } else {
        const T y = w * k;
        const T a0 = ST == 0 ? E * xn : acc;
        const T sm = a0 + y;
        const T bb = sm - a0;
        const T e = (a0 - (sm - bb)) + (y - bb);
        const T l = (ST == 0 ? E * err : lo) + e;
        if constexpr (ST != 3) {
            acc_out = sm;
            lo_out = l;
            return cn * xn + an * k;
        }
        const T x = sm + l;
        err_out = l - (x - sm);
        return x;
    }
}

// Increments of the auxiliaries' stage values over Q_n at the point and the neighbours the
// layer terms read.
template <typename T> struct RkE { T u0, ui, uk, v0, vj, vk, w0, wk, p0, pi, pj, pk; };

// dt R of the four fields at the lane's point; xc: the stage state there.
template <typename T, int WM, bool TERRAIN, int ST, bool X, bool Y, bool Z>
__device__ __forceinline__ void rk_row_point(const RkRowArgs<T> &A, const RowGeo &G, const RowLane &l, const RowPos &ps, int k,
                                             const RowLine<T> &yl, const RowLine<T> &zl, const RowSlab<T> &sy,
                                             const RowSlab<T> &sz, T (&xc)[4], T (&kf)[4])
{
    const AirArgs<T> &a = A.a;
    const Grid<T> &g = a.g;
    const size_t snx = (size_t)G.nx * sizeof(T), sxy = snx * G.ny;
    const unsigned op = ps.op, ox = (unsigned)l.ip * (unsigned)sizeof(T);
    const RowAt<T> at{snx * ps.jb + sxy * k, snx, sxy, op};
    Nb<T> n;
    row_metric<T, TERRAIN>(row_column<T, TERRAIN>(g, G.nx, l.ip, ps.jb, op), yl.m, zl.m, zl.t, n);
    Lay<T> lx{}, ly{}, lz{};
    QP<T> px{}, py{}, pz{};
    QV<T> vx{}, vy{}, vz{};
    RkE<T> e{};
    if constexpr (ST != 0 && (X || Y || Z)) {
        const T dt = g.dt, cp = A.cp;
        auto inc = [&](gptr<const T> f, int di, int dj, int dk) { return cp * (dt * at(f, di, dj, dk)); };
        gptr<const T> u = A.pv[0], v = A.pv[1], w = A.pv[2], p = A.pv[3];
        e.u0 = inc(u, 0, 0, 0); e.ui = inc(u, 1, 0, 0);
        e.v0 = inc(v, 0, 0, 0); e.vj = inc(v, 0, 1, 0);
        e.w0 = inc(w, 0, 0, 0); e.wk = inc(w, 0, 0, 1);
        e.p0 = inc(p, 0, 0, 0); e.pi = inc(p, -1, 0, 0); e.pj = inc(p, 0, -1, 0); e.pk = inc(p, 0, 0, -1);
        if constexpr (TERRAIN) { e.uk = inc(u, 0, 0, 1); e.vk = inc(v, 0, 0, 1); }
    }
    // a stage value of the auxiliaries: Q_n and its increment
    auto s = [&](T q, T d) {
        if constexpr (ST == 0) return q;
        else return q + d;
    };
    if constexpr (X) {
        const RowX q = row_x<T>(G, l.ip, ps.j, k);
        const RowQ<T> &Q = A.q[0];
        lx = {ldr<T>(A.xs, 0, ox), ldr<T>(A.xc, 0, ox), (Y || Z) ? ldr<T>(A.xd, 0, ox) : T(0), q.act};
        px.v0 = s(ldr<T>(Q.o[1], 0, q.o), e.v0); px.vj = s(ldr<T>(Q.o[1], 0, q.o + q.dj), e.vj);
        px.w0 = s(ldr<T>(Q.o[2], 0, q.o), e.w0); px.wk = s(ldr<T>(Q.o[2], 0, q.o + q.dk), e.wk);
        if constexpr (TERRAIN) px.vk = s(ldr<T>(Q.o[1], 0, q.o + q.dk), e.vk);
        vx.p0 = s(ldr<T>(Q.o[3], 0, q.o), e.p0); vx.pj = s(ldr<T>(Q.o[3], 0, q.o - q.dj), e.pj);
        vx.pk = s(ldr<T>(Q.o[3], 0, q.o - q.dk), e.pk);
        if constexpr (Y || Z) {
            px.u0 = s(ldr<T>(Q.o[0], 0, q.o), e.u0); px.ui = s(ldr<T>(Q.o[0], 0, q.o + q.di), e.ui);
            if constexpr (TERRAIN) px.uk = s(ldr<T>(Q.o[0], 0, q.o + q.dk), e.uk);
            vx.pi = s(ldr<T>(Q.o[3], 0, q.o - q.di), e.pi);
            px.p0 = vx.p0;
            vx.u0 = px.u0; vx.v0 = px.v0; vx.w0 = px.w0;
        }
    }
    if constexpr (Y) {
        const RowQ<T> &Q = A.q[1];
        ly = {sy.s, sy.c, sy.d, sy.act};
        py.u0 = s(ldr<T>(Q.o[0], sy.row, op), e.u0); py.ui = s(ldr<T>(Q.o[0], sy.row, op, sizeof(T)), e.ui);
        py.w0 = s(ldr<T>(Q.o[2], sy.row, op), e.w0); py.wk = s(ldr<T>(Q.o[2], sy.row + sy.dk, op), e.wk);
        if constexpr (TERRAIN) py.uk = s(ldr<T>(Q.o[0], sy.row + sy.dk, op), e.uk);
        vy.p0 = s(ldr<T>(Q.o[3], sy.row, op), e.p0); vy.pi = s(ldr<T>(Q.o[3], sy.row, op, -(int)sizeof(T)), e.pi);
        vy.pk = s(ldr<T>(Q.o[3], sy.row - sy.dk, op), e.pk);
        if constexpr (Z) {
            py.v0 = s(ldr<T>(Q.o[1], sy.row, op), e.v0); py.vj = s(ldr<T>(Q.o[1], sy.row + sy.dj, op), e.vj);
            if constexpr (TERRAIN) py.vk = s(ldr<T>(Q.o[1], sy.row + sy.dk, op), e.vk);
            vy.pj = s(ldr<T>(Q.o[3], sy.row - sy.dj, op), e.pj);
            py.p0 = vy.p0;
            vy.u0 = py.u0; vy.v0 = py.v0; vy.w0 = py.w0;
        }
    }
    if constexpr (Z) {
        const RowQ<T> &Q = A.q[2];
        lz = {sz.s, sz.c, sz.d, sz.act};
        pz.u0 = s(ldr<T>(Q.o[0], sz.row, op), e.u0); pz.ui = s(ldr<T>(Q.o[0], sz.row, op, sizeof(T)), e.ui);
        pz.v0 = s(ldr<T>(Q.o[1], sz.row, op), e.v0); pz.vj = s(ldr<T>(Q.o[1], sz.row + sz.dj, op), e.vj);
        if constexpr (TERRAIN) {
            pz.uk = s(ldr<T>(Q.o[0], sz.row + sz.dk, op), e.uk);
            pz.vk = s(ldr<T>(Q.o[1], sz.row + sz.dk, op), e.vk);
        }
        vz.p0 = s(ldr<T>(Q.o[3], sz.row, op), e.p0); vz.pi = s(ldr<T>(Q.o[3], sz.row, op, -(int)sizeof(T)), e.pi);
        vz.pj = s(ldr<T>(Q.o[3], sz.row - sz.dj, op), e.pj);
        if constexpr (TERRAIN) vz.pk = s(ldr<T>(Q.o[3], sz.row - sz.dk, op), e.pk);
    }
    T ddx, ddy, dwz, gpx, gpy, gpz;
    const RowState<T> st{g, at};
    T r = row_dp<T, WM, TERRAIN, true>(a, at, st, n, ddx, ddy, dwz);
    kf[3] = row_dp_layers<T, TERRAIN, X, Y, Z>(a, n, lx, ly, lz, px, py, pz, n.pc, ddx, ddy, dwz, r);
    T du, dv, dw;
    row_duvw<T, WM, TERRAIN, true>(a, at, st, n, gpx, gpy, gpz, du, dv, dw);
    row_duvw_layers<T, TERRAIN, X, Y, Z>(a, n, lx, ly, lz, vx, vy, vz, n.uc, n.vc, n.wc, gpx, gpy, gpz, du, dv, dw);
    kf[0] = du; kf[1] = dv; kf[2] = dw;
    xc[0] = n.uc; xc[1] = n.vc; xc[2] = n.wc; xc[3] = n.pc;
}

// The auxiliaries of node i of row (j, k) at level n+1, from Q_n and the node's states of the
// four stages (read before anything is stored; RkAux holds them until then).
template <typename T> struct RkAux {
    RowX x;
    RowSlab<T> y, z;
    unsigned o;
    T q[3][4];
};
template <typename T>
__device__ __forceinline__ void rk_aux_read(const RkRowArgs<T> &A, const RowGeo &G, const RowLine<T> &yl, const RowLine<T> &zl, int i,
                                            const RowPos &ps, int k, RkAux<T> &r)
{
    const unsigned o = r.o = ps.on;
    const size_t row = (size_t)G.nx * ((size_t)ps.jb + (size_t)G.ny * k) * sizeof(T);
    r.x = row_x<T>(G, i, ps.j, k);
    r.y = row_slab_y(yl, G.nx, k);
    r.z = row_slab_z(zl, G.nx, G.ny, ps.jb);
    if (!r.x.own && !r.y.in && !r.z.in) return;
    const T dt = A.a.g.dt;
    gptr<const T> c[4] = {A.a.g.un, A.a.g.vn, A.a.g.wn, A.a.g.pn};
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        T qx = T(0), qy = T(0), qz = T(0);
        if (r.x.own) qx = ldr<T>(A.q[0].o[f], 0, r.x.o);
        if (r.y.in) qy = ldr<T>(A.q[1].o[f], r.y.row, o);
        if (r.z.in) qz = ldr<T>(A.q[2].o[f], r.z.row, o);
        const T y0 = ldr<T>(A.xn[f], row, o), y1 = ldr<T>(A.y1[f], row, o), y2 = ldr<T>(A.pv[f], row, o), y3 = ldr<T>(c[f], row, o);
        const T b0 = rk_w<T, 0>() * (dt * y0), b1 = rk_w<T, 1>() * (dt * y1), b2 = rk_w<T, 1>() * (dt * y2), b3 = rk_w<T, 3>() * (dt * y3);
        r.q[0][f] = (((qx + b0) + b1) + b2) + b3;
        r.q[1][f] = (((qy + b0) + b1) + b2) + b3;
        r.q[2][f] = (((qz + b0) + b1) + b2) + b3;
    }
}
template <typename T> __device__ __forceinline__ void rk_aux_write(const RkRowArgs<T> &A, const RkAux<T> &r)
{
    const unsigned o = r.o;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        if (r.x.own) str<T>(A.q[0].n[f], 0, r.x.o, r.q[0][f]);
        if (r.y.in) str<T>(A.q[1].n[f], r.y.row, o, r.q[1][f]);
        if (r.z.in) str<T>(A.q[2].n[f], r.z.row, o, r.q[2][f]);
    }
}

template <typename T> __device__ __forceinline__ void rk_store4(gptr<T> const (&f)[4], size_t row, unsigned o, const T (&v)[4])
{
#pragma unroll
    for (int c = 0; c < 4; ++c) str<T>(f[c], row, o, v[c]);
}
// A face node of the air: the destination state and, in the last stage, its auxiliaries.
template <typename T, int ST>
__device__ __forceinline__ void rk_node(const RkRowArgs<T> &A, const RowGeo &G, int i, int j, int k, const T (&v)[4])
{
    const size_t row = (size_t)G.nx * ((size_t)j + (size_t)G.ny * k) * sizeof(T);
    const unsigned o = (unsigned)i * (unsigned)sizeof(T);
    if constexpr (ST == 3) {
        RkAux<T> r;
        rk_aux_read(A, G, row_line(A.yl, j), row_line(A.zl, k), i, RowPos{j, j, o, o}, k, r);
        rk_store4(A.dst, row, o, v);
        rk_aux_write(A, r);
    } else {
        rk_store4(A.dst, row, o, v);
    }
}
template <typename T> __device__ __forceinline__ void rk_pore_node(const RkRowArgs<T> &A, const RowGeo &G, int i, int j, int k, const T (&v)[4])
{
    rk_store4(A.pdst, (size_t)G.nx * ((size_t)j + (size_t)G.ny * k) * sizeof(T), (unsigned)i * (unsigned)sizeof(T), v);
}

// Destination state of a porous point (rk_pore_point of the general form): dt R_p = -gama div u
// (porous.cpp:77-95), dt R_u = -dt eff grad p with the drag in the integrating factor.
template <typename T, bool TERRAIN, int ST>
__device__ __forceinline__ void rk_row_pore(const RkRowArgs<T> &A, const RowGeo &G, int st, const RowLane &l, int j, int k, T (&d)[4])
{
    constexpr bool COMP = std::is_same<T, float>::value;
    const Grid<T> &g = A.pore;
    const size_t snx = (size_t)G.nx * sizeof(T), sxy = snx * G.ny;
    const unsigned op = (unsigned)l.ip * (unsigned)sizeof(T);
    const RowAt<T> at{snx * j + sxy * k, snx, sxy, op};
    Nb<T> n;
    row_metric<T, TERRAIN>(g, G.nx, l.ip, j, lds_<T>(g.my, j), lds_<T>(g.mz, k), TERRAIN ? lds_<T>(g.ttk, k) : T(0), n);
    T xc[4] = {at(g.un, 0, 0, 0), at(g.vn, 0, 0, 0), at(g.wn, 0, 0, 0), at(g.pn, 0, 0, 0)};
    T xn[4], ac[4], lo[4], er[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        xn[f] = ST == 0 ? xc[f] : ST == 3 && !COMP ? T(0) : at(A.pxn[f], 0, 0, 0);
        ac[f] = ST != 0 ? at(A.pacc[f], 0, 0, 0) : T(0);
        lo[f] = COMP && ST != 0 && f < 3 ? at(A.plo[f], 0, 0, 0) : T(0);
        er[f] = COMP && ((ST == 0 && f < 3) || (ST == 3 && f == 3)) ? at(A.perr[f], 0, 0, 0) : T(0);
    }
    const T dux = at(g.un, 1, 0, 0) - xc[0], dvy = at(g.vn, 0, 1, 0) - xc[1], dwz = at(g.wn, 0, 0, 1) - xc[2];
    T div;
    if constexpr (TERRAIN) {
        const T duz = at(g.un, 0, 0, 1) - xc[0], dvz = at(g.vn, 0, 0, 1) - xc[1];
        div = (((((n.mX * g.dxi) * dux) + ((n.zX * g.dzi) * duz)) + ((n.mY * g.dyi) * dvy)) + ((n.zY * g.dzi) * dvz)) +
              ((n.mZ * g.dzi) * dwz);
    } else {
        div = (((n.mX * g.dxi) * dux) + ((n.mY * g.dyi) * dvy)) + ((n.mZ * g.dzi) * dwz);
    }
    T gx, gy, gz;
    row_pore_grad<T, TERRAIN>(g, at, n, g.pn, gx, gy, gz);
    const T f = (-g.dt) * A.peff;
    const T kf[4] = {f * gx, f * gy, f * gz, (-A.pgama) * div};
    T ao[4], lw[4], eo[4];
    const T cf[5] = {A.cf[0], A.cf[1], A.cf[2], A.cf[3], A.cf[4]};
#pragma unroll
    for (int q = 0; q < 3; ++q) d[q] = rk_point_if<T, ST>(st, xn[q], kf[q], ac[q], lo[q], er[q], cf, ao[q], lw[q], eo[q]);
    d[3] = rk_point<T, ST>(xn[3], kf[3], ac[3], er[3], A.ca, ao[3], eo[3]);
    if (!l.live || l.face) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if constexpr (ST != 3) {
            str<T>(A.pacc[q], at.row, op, ao[q]);
            if (COMP && q < 3) str<T>(A.plo[q], at.row, op, lw[q]);
        } else if constexpr (COMP) {
            str<T>(A.perr[q], at.row, op, eo[q]);
        }
    }
}

// The air point of a lane: registers, stencil, stores of its node (d: the destination state).
// YS: the row may lie in a y layer.
template <typename T, int WM, bool TERRAIN, int ST, bool YS>
__device__ __forceinline__ void rk_row_air(const RkRowArgs<T> &A, const RowGeo &G, const RowLane &l, const RowPos &ps, int k,
                                           const RowLine<T> &yl, const RowLine<T> &zl, bool mx, T (&d)[4])
{
    constexpr bool COMP = std::is_same<T, float>::value;
    const int nx = G.nx, ny = G.ny;
    const RowSlab<T> sy = row_slab_y(yl, nx, k), sz = row_slab_z(zl, nx, ny, ps.jb);
    const size_t row = (size_t)nx * ((size_t)ps.jb + (size_t)ny * k) * sizeof(T);
    const unsigned op = ps.op;
    const size_t e = (size_t)l.ip + (size_t)nx * ((size_t)ps.j + (size_t)ny * k);
    // the point's registers, the auxiliaries of the last stage, then the stencil
    T xn[4], ac[4] = {T(0), T(0), T(0), T(0)}, er[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        xn[f] = ST == 0 || (ST == 3 && !COMP) ? T(0) : ldr<T>(A.xn[f], row, op);
        er[f] = ST == 3 && COMP ? ldr<T>(A.err[f], row, op) : T(0);
    }
    if constexpr (ST != 0) acc4_load(A.acc, e, ac);
    T xc[4], kf[4];
#define LEE_BODY(X, Y, Z) rk_row_point<T, WM, TERRAIN, ST, X, Y, Z>(A, G, l, ps, k, yl, zl, sy, sz, xc, kf)
    if (!sz.in) {
        if (!YS || !sy.in) { if (mx) LEE_BODY(true, false, false); else LEE_BODY(false, false, false); }
        else { if (mx) LEE_BODY(true, YS, false); else LEE_BODY(false, YS, false); }
    } else {
        if (!YS || !sy.in) { if (mx) LEE_BODY(true, false, true); else LEE_BODY(false, false, true); }
        else { if (mx) LEE_BODY(true, YS, true); else LEE_BODY(false, YS, true); }
    }
#undef LEE_BODY
    T ao[4], eo[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) d[f] = rk_point<T, ST>(ST == 0 ? xc[f] : xn[f], kf[f], ac[f], er[f], A.ca, ao[f], eo[f]);
    if (l.face) d[0] = T(0);
    if (l.live) {
        RkAux<T> r;
        if constexpr (ST == 3) rk_aux_read(A, G, yl, zl, l.in, ps, k, r);
        rk_store4(A.dst, row, ps.on, d);
        if (!l.face) {
            if constexpr (ST != 3) acc4_store(A.acc, e, ao);
            if constexpr (ST == 3 && COMP) {
#pragma unroll
                for (int f = 0; f < 4; ++f) str<T>(A.err[f], row, op, eo[f]);
            }
        }
        if constexpr (ST == 3) rk_aux_write(A, r);
    }
}

// MODE 1: a domain (box: the interior its ring's tiles leave out, or empty), 2: an ensemble's.
template <typename T, int WM, bool TERRAIN, int ST, int MODE>
__device__ __forceinline__ void rk_row_block(const RkRowArgs<T> &A, int st, int kind, int k, int tx, int ty, long long rec,
                                             double *__restrict__ rec_out, T (&rows)[RY][RX], const int (&box)[4])
{
    const RowGeo G = A.geo;
    const int nx = G.nx, ny = G.ny, nz = G.nz;
    const int lane = threadIdx.x, tj = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    if (ST == 0 && MODE != 2 && kind == RK_REC) {
        // receivers sample level n before the step (airpore.cpp:573-580)
        const long long r = rec * (RX * RY) + tj * RX + lane;
        if (r < G.nrec) {
            const long long q = A.rec_idx[r];
            double v = q >= 0 ? (double)A.a.g.pn[q] : 0.0;
            if (fabs(v) < 1.0e-100) v = 0.0;
            rec_out[r] = v;
        }
        return;
    }
    const int jr = G.j0 + RY * ty + tj;
    const bool row_live = jr >= 1;
    const int j = row_live ? jr : 1;
    const int i0 = G.i0 + tx * RX;
    RowLane l = row_lane(i0 + lane, nx, row_live);
    const bool last = ty == G.nty - 1;
    if (MODE == 1 && j >= box[2] && j < box[3]) {
        // the interior's points [box 0, box 1) of this row belong to its own kernel: their lanes
        // repeat the nearest other point (a tile never meets both ends of the interior)
        if (i0 >= box[0] && i0 + RX <= box[1]) return;  // (never in the last tile row)
        if (l.in >= box[0] && l.in < box[1]) l.live = false;
        l.ip = i0 < box[0] ? min(l.ip, box[0] - 1) : max(l.ip, box[1]);
    }
    T d[4];
    if (kind == RK_AIR) {
        rk_row_air<T, WM, TERRAIN, ST, true>(A, G, l, row_pos<T>(l, j), k, row_line(A.yl, j), row_line(A.zl, k), row_meets_x(G, i0), d);
    } else {
        rk_row_pore<T, TERRAIN, ST>(A, G, st, l, j, k, d);
        if (l.face) d[0] = T(0);
        if (l.live) rk_pore_node(A, G, l.in, j, k, d);
    }
    T pe = T(0);
    if (last) {
        rows[tj][lane] = d[3];
        __syncthreads();
        if (jr == ny - 2) pe = T(15.0 / 8.0) * d[3] - T(5.0 / 4.0) * rows[tj - 1][lane] + T(3.0 / 8.0) * rows[tj - 2][lane];
    }
    if (!l.live) return;
    const bool top = kind == RK_AIR && k == nz - 2, floor = kind == RK_AIR && k == 1;
    const bool pore_top = kind == RK_PORE && k == G.pnz - 2, pore_low = kind == RK_PORE && k == 1;
    if (jr != 1 && jr != ny - 2 && !top && !floor && !pore_top && !pore_low) return;
#pragma unroll 1
    for (int c = 0; c < 3; ++c) {
        if (c == 1 && jr != 1) continue;
        if (c == 2 && jr != ny - 2) continue;
        const int jn = c == 0 ? j : c == 1 ? 0 : ny - 1;
        const T v[4] = {d[0], c == 0 ? d[1] : T(0), d[2], c == 2 ? pe : d[3]};
        const T v0[4] = {v[0], v[1], T(0), v[3]};  // on a rigid horizontal face
        if (kind == RK_PORE) {
            if (c) rk_pore_node(A, G, l.in, jn, k, v);
            if (pore_low) rk_pore_node(A, G, l.in, jn, 0, v0);
            if (pore_top) rk_node<T, ST>(A, G, l.in, jn, 0, v);
        } else {
            if (c) rk_node<T, ST>(A, G, l.in, jn, k, v);
            if (top) rk_node<T, ST>(A, G, l.in, jn, nz - 1, v0);
            if (floor) {
                if (G.porous) rk_pore_node(A, G, l.in, jn, G.pnz - 1, v);
                else rk_node<T, ST>(A, G, l.in, jn, 0, v0);
            }
        }
    }
}

// A strip's block: 4 x S.rows rows from block row `br`, S.rows of them per wavefront, without a face
// in y or z (row_plan).  Waves of mostly idle lanes cost as much as full ones: the time of these
// kernels goes by waves (loads, waits and scalar work each) before it goes by bytes.  us per step
// before -> after: 137 x 91 x 53 FP64 (rows of 64 + 64 + 9) 196 -> 176, 512 x 256 x 128 (an interior
// leaves 21 columns of the outer tiles) FP32 1570 -> 1532, FP64 3046 -> 2838, 768 x 384 x 192 FP32
// (25 columns, two rows a wave) 4217 -> 4140.  Strips wider than a third of a wave at a row's end
// did not pay (160 = 64 + 64 + 32 columns: 3 % slower).  Also tried: a plane's blocks padded to
// eights (fewer bytes on small grids, 1-5 % slower on the others) and an eighth of the rows to each
// XCD (4 % slower in FP32), and half the waves for the pressure, half for the velocities (less than
// half the registers, 3 instead of 2 waves a SIMD in FP64, and 1.15-1.3 times the time).
template <typename T, int WM, bool TERRAIN, int ST>
__device__ __forceinline__ void rk_row_strip(const RkRowArgs<T> &A, const RowStrip &S, int ja, int je, int k, int br)
{
    const RowGeo G = A.geo;
    RowLane l;
    RowPos ps;
    if (!row_strip<T>(S, ja, je, br, G.nx, l, ps)) return;
    RowLine<T> yl{};
    yl.m = ldr<T>(A.a.g.my, 0, (unsigned)ps.j * (unsigned)sizeof(T));
    T d[4];
    rk_row_air<T, WM, TERRAIN, ST, false>(A, G, l, ps, k, yl, row_line(A.zl, k), S.x0 < G.xa || S.x0 + S.n > G.xb, d);
}

// q / d and the remainder from m = 2^32 / d (rounded up; one too large at most).
__device__ __forceinline__ int row_div(int q, int d, unsigned m, int &rem)
{
    int n = (int)__umulhi((unsigned)q, m);
    rem = q - n * d;
    if (rem < 0) { --n; rem += d; }
    if (rem >= d) { ++n; rem -= d; }
    return n;
}
// Block b of a launch: its section (planes below ka, above kb, the listed blocks of those between,
// porous layer, receivers), plane and tile.  Without strips or an interior the launch is a grid of
// tiles and planes instead, which spares the divisions (3 % on 160 x 96 x 64).
template <typename T, int WM, bool TERRAIN, int ST, int MODE>
__device__ __forceinline__ void rk_row_any(const RkRowArgs<T> &A, const RowLaunch &L, int b, int st, double *__restrict__ rec_out)
{
    __shared__ T rows[RY][RX];
    int box[4] = {0, 0, 0, 0}, idx, k, tx, ty, kind = RK_AIR, f = 0;
    if (MODE == 1 && L.grid) {
        const int z = blockIdx.z;
        tx = blockIdx.x; ty = blockIdx.y;
        kind = z < L.zair ? RK_AIR : z < L.zair + L.zpore ? RK_PORE : RK_REC;
        k = kind == RK_AIR ? z + 1 : z - L.zair + 1;
        b = ((z - L.zair - L.zpore) * L.nty + ty) * L.ntx + tx;
    } else if (b >= L.first[2] && b < L.first[3]) {
        k = L.ka + row_div(b - L.first[2], L.nring, L.by_ring, idx);
        const int e = ((const __attribute__((address_space(4))) int *)L.ring)[idx];
        if (e & kStripBlock) {
            const bool hi = e & (1 << 20);
            const RowStrip S{hi ? L.strip[1].x0 : L.strip[0].x0, hi ? L.strip[1].n : L.strip[0].n,
                             hi ? L.strip[1].rows : L.strip[0].rows, hi ? L.strip[1].inv : L.strip[0].inv};
            rk_row_strip<T, WM, TERRAIN, ST>(A, S, L.ja, L.jb, k, e & 0xfffff);
            return;
        }
        tx = e & 0xffff; ty = e >> 16;
        box[0] = L.xa; box[1] = L.xb; box[2] = L.ya; box[3] = L.yb;
    } else {
        int k0 = 1;
        if (b >= L.first[1]) { f = L.first[1]; k0 = L.kb; }
        if (b >= L.first[3]) { f = L.first[3]; k0 = 1; kind = RK_PORE; }
        if (b >= L.first[5]) { f = L.first[5]; kind = RK_REC; }
        k = k0 + row_div(b - f, L.ntx * L.nty, L.by_full, idx);
        ty = row_div(idx, L.ntx, L.by_ntx, tx);
    }
    rk_row_block<T, WM, TERRAIN, ST, MODE>(A, st, kind, k, tx, ty, b - f, rec_out, rows, box);
}
template <typename T, int WM, bool TERRAIN, int ST>
__global__ __launch_bounds__(RX * RY) void k_rk_row(const RkRowArgs<T> *__restrict__ ap, RowLaunch L, int st, double *__restrict__ rec_out)
{
    rk_row_any<T, WM, TERRAIN, ST, 1>(*ap, L, (int)blockIdx.x, st, rec_out);
}
// Ensemble: the members' arguments one after the other, the member of each block from a table (a
// search over the members' first blocks cost five dependent loads per wavefront).
template <typename T, int WM, bool TERRAIN, int ST>
__global__ __launch_bounds__(RX * RY) void k_rk_row_batch(const RkRowArgs<T> *__restrict__ ap, const int *__restrict__ member, int st)
{
    const RkRowArgs<T> &A = ap[((const __attribute__((address_space(4))) int *)member)[blockIdx.x]];
    rk_row_any<T, WM, TERRAIN, ST, 2>(A, A.whole, (int)blockIdx.x - A.first, st, nullptr);
}

// ---- the interior outside every layer and away from every face: two stages per launch ------
// A stage of the interior reads and writes 13 to 25 words a point at 4.2 of the 4.7 TB/s a copy
// reaches, so only fewer passes make it faster.  Here a block marches up its columns and keeps
// stage s's state y of four planes in LDS: plane k + 1 of y from the state in memory, then stage
// s + 1 of plane k from y.  Two stages move 13 + 25 words (FP32; 13 + 17 in FP64) instead of 34 +
// 46 (34 + 34).  Per step, 512 x 256 x 128 with wind over a hill: the interior 702 us by single
// stages (8.8 M points, whole tiles) and 578 us so (10.7 M points, any), the step 1779 -> 1570 us in
// FP32 and 3476 -> 3046 us in FP64; 768 x 384 x 192 FP32 4860 -> 4217 us.  At 2.7 to 3.5 TB/s it is
// bound by the latency of its loads and the barrier between the stages.  The y around a block's columns is computed by the neighbours as well; next to the
// interior it is read from the buffer stage s left it in, and the interior's outermost points
// store theirs there for the ring's stage s + 1.
//
// The lane's own column (state, mean flow along y, and in the second pair level n, accumulator
// and error) is loaded a plane ahead into registers, so that loads from memory are in flight all
// through a plane.  Loads and stores are waited for in order, so the neighbours' values of the
// next plane, which the caches hold by then, are requested before stage s + 1 stores.  Without the
// column loaded ahead the pairs took 741 us (FP32) and 1182 us (FP64: 1002 us so), with the
// neighbours requested after the column's next plane 655 us, after the stores 580 us; FP32 blocks
// of 8 rows 635 us; nontemporal stores the same as plain ones.
template <typename T> constexpr int kPR = pair_rows(sizeof(T));  // rows of a block with the two around its own

// Readers around the lane's point: the state with the lane's column and its four neighbours (x + 1,
// x - 1, y + 1, y - 1) in registers, ...
template <typename T> struct PairColumn {
    const T (&r)[3][4], (&nb)[4][4];
    template <int C> __device__ __forceinline__ T get(int di, int dj, int dk) const
    {
        constexpr int f = C > 3 ? 3 : C;
        return di ? nb[di > 0 ? 0 : 1][f] : dj ? nb[dj > 0 ? 2 : 3][f] : r[dk + 1][f];
    }
};
// ... the mean flow (V alone: in registers too), ...
template <typename T, int WM> struct PairWind {
    const RowAt<T> &at;
    const T *r, *nb;
    __device__ __forceinline__ T operator()(gptr<const T> f, int di, int dj, int dk) const
    {
        if constexpr (WM == 2) return di ? nb[di > 0 ? 0 : 1] : dj ? nb[dj > 0 ? 2 : 3] : r[dk + 1];
        else return at(f, di, dj, dk);
    }
};
// ... and y from LDS planes k - 1, k, k + 1.
template <typename T> struct PairState {
    const T *y[3];  // the lane's value of field 0
    template <int C> __device__ __forceinline__ T get(int di, int dj, int dk) const
    {
        return y[dk + 1][(C > 3 ? 3 : C) * kPR<T> * RX + dj * RX + di];
    }
};
template <typename T> struct PairPoint {
    T xn[4], acc[4];  // level n, accumulator after stage s
    T V[4];           // mean flow at the four neighbours
};

template <typename T, int WM, bool TERRAIN, bool LAST>
__global__ __launch_bounds__(RX * kPR<T>) void k_rk_pair(const RkRowArgs<T> *__restrict__ ap, RowPair bx)
{
    constexpr bool COMP = std::is_same<T, float>::value;
    constexpr int SA = LAST ? 1 : 0, SB = LAST ? 3 : 1;
    __shared__ T Y[4][4][kPR<T>][RX];
    const RkRowArgs<T> &A = ap[0], &B = ap[1];
    const AirArgs<T> &a = A.a;
    const Grid<T> &g = a.g;
    const int lane = threadIdx.x, row = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    // blocks that follow one another in a plane share an XCD (and the columns around them its L2)
    const int blocks = gridDim.x, b = blockIdx.x, xcd = b & 7, per = blocks >> 3, more = blocks & 7;
    const int t = xcd * per + min(xcd, more) + (b >> 3);
    const int plane = bx.nbx * bx.nby, tz = t / plane, tp = t - tz * plane, ty = tp / bx.nbx, tx = tp - ty * bx.nbx;
    const int x0 = bx.xa + tx * bx.wx, x1 = min(x0 + bx.wx, bx.xb), y0 = bx.ya + ty * bx.wy, y1 = min(y0 + bx.wy, bx.yb);
    const int k0 = bx.za + tz * bx.wz, k1 = min(k0 + bx.wz, bx.zb);
    // lanes and rows past the block's last repeat the one after it
    const int i = min(x0 - 1 + lane, x1), j = min(y0 - 1 + row, y1);
    const bool own = lane >= 1 && x0 - 1 + lane < x1 && row >= 1 && y0 - 1 + row < y1;
    const bool in = i >= bx.xa && i < bx.xb && j >= bx.ya && j < bx.yb;
    const bool rim = i == bx.xa || i == bx.xb - 1 || j == bx.ya || j == bx.yb - 1;
    const size_t snx = (size_t)g.nx * sizeof(T), sxy = snx * g.ny;
    const unsigned o = (unsigned)i * (unsigned)sizeof(T);
    auto at_plane = [&](int k) { return RowAt<T>{snx * j + sxy * k, snx, sxy, o}; };
    auto elem = [&](int k) { return (size_t)i + (size_t)g.nx * ((size_t)j + (size_t)g.ny * k); };
    // planes k - 1, k, k + 1 of the state, k - 2 .. k + 1 of V; level n, accumulator of plane k,
    // error of plane k - 1
    T r[3][4], v[4] = {}, xn[4] = {}, ac[4] = {}, er[4] = {};
    T r2[4], v2 = T(0), xn2[4] = {}, ac2[4] = {}, er2[4] = {};  // the next plane's
    const RowColumn<T> col = row_column<T, TERRAIN>(g, g.nx, i, j, o);
    const T my = lds_<T>(g.my, j);
    auto column = [&](int k, T(&q)[4]) {
        const RowAt<T> at = at_plane(k);
        q[0] = at(g.un, 0, 0, 0); q[1] = at(g.vn, 0, 0, 0); q[2] = at(g.wn, 0, 0, 0); q[3] = at(g.pn, 0, 0, 0);
    };
    auto level = [&](int k, T(&q)[4]) {
        const RowAt<T> at = at_plane(k);
#pragma unroll
        for (int f = 0; f < 4; ++f) q[f] = at(A.xn[f], 0, 0, 0);
    };
    column(k0 - 2, r[1]);
    column(k0 - 1, r[2]);
    column(k0, r2);
    if constexpr (WM == 2) {
        v[2] = at_plane(k0 - 2)(a.V, 0, 0, 0);
        v[3] = at_plane(k0 - 1)(a.V, 0, 0, 0);
        v2 = at_plane(k0)(a.V, 0, 0, 0);
    }
    if constexpr (LAST) level(k0 - 1, xn2);
    // the neighbours' values of plane k, or the plane's own y outside the interior
    T nb[4][4] = {}, vn[4] = {};
    auto inside = [&](int k) { return in && k >= bx.za && k < bx.zb; };
    auto neighbours = [&](int k) {
        const RowAt<T> at = at_plane(k);
        if (inside(k)) {
            constexpr int D[4][2] = {{1, 0}, {-1, 0}, {0, 1}, {0, -1}};
            const RowState<T> st{g, at};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                nb[q][0] = st.template get<0>(D[q][0], D[q][1], 0);
                nb[q][1] = st.template get<1>(D[q][0], D[q][1], 0);
                nb[q][2] = st.template get<2>(D[q][0], D[q][1], 0);
                nb[q][3] = st.template get<3>(D[q][0], D[q][1], 0);
                if constexpr (WM == 2) vn[q] = at(a.V, D[q][0], D[q][1], 0);
            }
        } else {
            nb[0][0] = at(A.dst[0], 0, 0, 0); nb[1][3] = at(A.dst[1], 0, 0, 0);
            nb[2][1] = at(A.dst[2], 0, 0, 0); nb[3][3] = at(A.dst[3], 0, 0, 0);
        }
    };
    neighbours(k0 - 1);
    PairPoint<T> c{}, n{};
#pragma unroll 1
    for (int k = k0 - 1; k <= k1; ++k) {
        const RowAt<T> at = at_plane(k);
        T y[4];
        // what the previous plane asked for, then the next plane's
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            r[0][f] = r[1][f]; r[1][f] = r[2][f]; r[2][f] = r2[f];
            xn[f] = xn2[f]; ac[f] = ac2[f]; er[f] = er2[f];
        }
        v[0] = v[1]; v[1] = v[2]; v[2] = v[3]; v[3] = v2;
        __builtin_amdgcn_sched_barrier(0);
        const int k2 = min(k + 2, k1 + 1), kn = min(k + 1, k1);
        column(k2, r2);
        if constexpr (WM == 2) v2 = at_plane(k2)(a.V, 0, 0, 0);
        if constexpr (LAST) {
            level(kn, xn2);
            if (own && kn < k1) acc4_load(A.acc, elem(kn), ac2);
            if constexpr (COMP) {
                const RowAt<T> ak = at_plane(min(k, k1 - 1));
                if (own && k >= k0)
#pragma unroll
                    for (int f = 0; f < 4; ++f) er2[f] = ak(B.err[f], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (inside(k)) {
            Nb<T> q;
            row_metric<T, TERRAIN>(col, my, lds_<T>(g.mz, k), TERRAIN ? lds_<T>(g.ttk, k) : T(0), q);
            T kf[4], ddx, ddy, dwz, gpx, gpy, gpz, e;
            const PairColumn<T> st{r, nb};
            const PairWind<T, WM> wind{at, v + 1, vn};
            kf[3] = row_dp<T, WM, TERRAIN, true>(a, wind, st, q, ddx, ddy, dwz);
            row_duvw<T, WM, TERRAIN, true>(a, wind, st, q, gpx, gpy, gpz, kf[0], kf[1], kf[2]);
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                n.xn[f] = LAST ? xn[f] : r[1][f];
                y[f] = rk_point<T, SA>(n.xn[f], kf[f], ac[f], T(0), A.ca, n.acc[f], e);
            }
            if (own && k >= k0 && k < k1 && (rim || k == bx.za || k == bx.zb - 1)) rk_store4(A.dst, at.row, o, y);
#pragma unroll
            for (int f = 0; f < 4; ++f) n.V[f] = vn[f];
        } else {
            y[0] = nb[0][0]; y[1] = nb[1][3]; y[2] = nb[2][1]; y[3] = nb[3][3];
        }
#pragma unroll
        for (int f = 0; f < 4; ++f) Y[k & 3][f][row][lane] = y[f];
        // the plane written next was last read before the previous barrier
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        neighbours(min(k + 1, k1));
        __builtin_amdgcn_sched_barrier(0);
        if (own && k > k0) {
            const int kc = k - 1;
            const RowAt<T> ac1 = at_plane(kc);
            Nb<T> q;
            row_metric<T, TERRAIN>(col, my, lds_<T>(g.mz, kc), TERRAIN ? lds_<T>(g.ttk, kc) : T(0), q);
            const PairState<T> st{{&Y[(kc - 1) & 3][0][row][lane], &Y[kc & 3][0][row][lane], &Y[(kc + 1) & 3][0][row][lane]}};
            const PairWind<T, WM> wind{ac1, v, c.V};
            T kf[4], ddx, ddy, dwz, gpx, gpy, gpz, d[4], ao[4], eo[4];
            kf[3] = row_dp<T, WM, TERRAIN, true>(a, wind, st, q, ddx, ddy, dwz);
            row_duvw<T, WM, TERRAIN, true>(a, wind, st, q, gpx, gpy, gpz, kf[0], kf[1], kf[2]);
#pragma unroll
            for (int f = 0; f < 4; ++f) d[f] = rk_point<T, SB>(c.xn[f], kf[f], c.acc[f], er[f], B.ca, ao[f], eo[f]);
            rk_store4(B.dst, ac1.row, o, d);
            if constexpr (!LAST) acc4_store(B.acc, elem(kc), ao);
            if constexpr (LAST && COMP) {
#pragma unroll
                for (int f = 0; f < 4; ++f) str<T>(B.err[f], ac1.row, o, eo[f]);
            }
        }
        c = n;
    }
}

}  // namespace

template <typename T>
void launch_rk_row(const RkRowArgs<T> *ad, const RowPlan &pl, int st, int wind, bool terrain, bool split, double *rec, hipStream_t s)
{
    const RowPair &bx = pl.pair;
    const RowLaunch &L = split ? st ? pl.v : pl.p : st ? pl.w[1] : pl.w[0];  // stage 0 with the receivers
    const dim3 blocks = L.grid ? dim3((unsigned)L.ntx, (unsigned)L.nty, (unsigned)L.z) : dim3((unsigned)L.first[6]);
#define LEE_RS(WM, TER, ST)                                                                                            \
    do {                                                                                                               \
        hipLaunchKernelGGL((k_rk_row<T, WM, TER, ST>), blocks, dim3(RX, RY), 0, s, ad, L, st, rec);                     \
        if (split && (st == 0 || st == 2))                                                                             \
            hipLaunchKernelGGL((k_rk_pair<T, WM, TER, ST != 0>), dim3((unsigned)(bx.nbx * bx.nby * bx.nbz)),            \
                               dim3(RX, kPR<T>), 0, s, ad, bx);                                                        \
    } while (0)
#define LEE_RT(WM, TER)                                                                            \
    do {                                                                                           \
        if (st == 0) LEE_RS(WM, TER, 0); else if (st == 3) LEE_RS(WM, TER, 3); else LEE_RS(WM, TER, 1); \
    } while (0)
    if (terrain) { if (wind == 1) LEE_RT(1, true); else if (wind == 2) LEE_RT(2, true); else LEE_RT(0, true); }
    else { if (wind == 1) LEE_RT(1, false); else if (wind == 2) LEE_RT(2, false); else LEE_RT(0, false); }
#undef LEE_RT
#undef LEE_RS
}
template <typename T>
void launch_rk_row_batch(const RkRowArgs<T> *ad, const int *member, int nblocks, int st, int wind, bool terrain, hipStream_t s)
{
    if (nblocks <= 0) return;
    const dim3 blk(RX, RY);
#define LEE_RS(WM, TER, ST) hipLaunchKernelGGL((k_rk_row_batch<T, WM, TER, ST>), dim3((unsigned)nblocks), blk, 0, s, ad, member, st)
#define LEE_RT(WM, TER)                                                                            \
    do {                                                                                           \
        if (st == 0) LEE_RS(WM, TER, 0); else if (st == 3) LEE_RS(WM, TER, 3); else LEE_RS(WM, TER, 1); \
    } while (0)
    if (terrain) { if (wind == 1) LEE_RT(1, true); else if (wind == 2) LEE_RT(2, true); else LEE_RT(0, true); }
    else { if (wind == 1) LEE_RT(1, false); else if (wind == 2) LEE_RT(2, false); else LEE_RT(0, false); }
#undef LEE_RT
#undef LEE_RS
}
template void launch_rk_row<LEE_RK_T>(const RkRowArgs<LEE_RK_T> *, const RowPlan &, int, int, bool, bool, double *, hipStream_t);
template void launch_rk_row_batch<LEE_RK_T>(const RkRowArgs<LEE_RK_T> *, const int *, int, int, int, bool, hipStream_t);

}  // namespace lee
