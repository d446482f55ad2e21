// lee_row.h -- row form of the air stencils: a wavefront takes 64 consecutive points of one row,
// so the row, the plane, the layers met along y and z and every row's base address are
// wave-uniform, and a field access is a scalar base plus the lane's 32-bit byte offset.
//
// What bounds the point kernels in the general form (lee_kernels.hip) is not HBM: a point of
// the layer shell went through 90-320 waits, one per slab and term, with 64-bit address
// arithmetic per access.  Here the slabs a wavefront can meet are template parameters
// (X, Y, Z), chosen by a scalar branch, and inside one instance there is no branch: every
// field and auxiliary of the point is read before the first store, one memory round trip per
// phase.  A layer term that does not apply (the outermost plane of a slab belongs to it for the
// auxiliaries only) is dropped by a select, so the sums are those of the general form bit for bit.
//
// Each axis must have its low and high slab apart (row_form in lee_ctx.hip); grids narrower
// than their layers, embedded obstacles and an uncoupled porous layer run the general form.
#pragma once

#include "lee_core.h"
#include "lee_kernels.h"

namespace lee {

namespace {

constexpr int RX = 64, RY = 4;  // points of a row per wavefront, rows per block

template <typename T> using gconst = const __attribute__((address_space(1))) T *;
template <typename T> __device__ __forceinline__ T ldr(gptr<const T> f, size_t row, unsigned o, int d = 0)
{
    return *(gconst<T>)((gconst<char>)f.p + row + (ptrdiff_t)d + o);
}
template <typename T> __device__ __forceinline__ void str(gptr<T> f, size_t row, unsigned o, T v)
{
    *(__attribute__((address_space(1))) T *)((__attribute__((address_space(1))) char *)f.p + row + o) = v;
}
// A value of a table at a wave-uniform index, as a scalar load.
template <typename T> __device__ __forceinline__ T lds_(gptr<const T> f, int i)
{
    return ((const __attribute__((address_space(4))) T *)f.p)[i];
}

// The rows of a block: tile row ty covers j0 + 4 ty .. + 3, anchored at the high end so that the
// last tile row holds the interior rows ny - 4, ny - 3, ny - 2 the East face's pressure is
// extrapolated from; rows below 1 of the first tile row idle (clamped to row 1, nothing stored).
inline int row_tiles(int ny) { return (ny - 2 + RY - 1) / RY; }
inline int row_first(int ny) { return ny - 1 - RY * row_tiles(ny); }
// x of a row's first lane: 0, or -1 where the last face would otherwise stand alone in its
// wavefront (the RK4 registers are updated in place, so the point a face lane computes must
// belong to its own wavefront).
inline int row_left(int nx) { return nx % RX == 1 ? -1 : 0; }

// Where a lane stands.  A lane on an x face (or past the row's end) computes the interior
// neighbour's point (ip) and stores it as its own node (in): the value the face's copy gives.
struct RowLane {
    int in, ip;           // node and point
    bool live;            // the node exists and the row is one of the interior's
    bool face;            // the node is on an x face
};
__device__ __forceinline__ RowLane row_lane(int i, int nx, bool row_live)
{
    RowLane l;
    l.in = i;
    l.ip = i < 1 ? 1 : i > nx - 2 ? nx - 2 : i;
    l.live = row_live && i >= 0 && i < nx;
    l.face = i == 0 || i == nx - 1;
    return l;
}

// Where a wavefront's lanes stand: a row jb (uniform) that addresses start from, the lane's row j
// (jb, or one of the next ones) and the byte offsets of its point and node from row jb's first.
struct RowPos {
    int jb, j;
    unsigned op, on;
};
template <typename T> __device__ __forceinline__ RowPos row_pos(const RowLane &l, int j)
{
    return {j, j, (unsigned)l.ip * (unsigned)sizeof(T), (unsigned)l.in * (unsigned)sizeof(T)};
}
// Lanes of block row `br` of a strip (four wavefronts, S.rows rows each); false: no row left.
template <typename T> __device__ __forceinline__ bool row_strip(const RowStrip &S, int ja, int je, int br, int nx, RowLane &l, RowPos &ps)
{
    const int lane = threadIdx.x, tj = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    const int jb = ja + (RY * br + tj) * S.rows;
    if (jb >= je) return false;
    int r = (lane * S.inv) >> 16;
    const int c = lane - r * S.n;
    const bool live = r < S.rows && jb + r < je;
    if (!live) r = 0;
    l = row_lane(S.x0 + c, nx, live);
    ps = {jb, jb + r, (unsigned)(l.ip + nx * r) * (unsigned)sizeof(T), (unsigned)(l.in + nx * r) * (unsigned)sizeof(T)};
    return true;
}

// The y or z layer of a row (wave-uniform): whether it lies in a slab, whether the layer terms
// apply, the byte offset of the row in the axis's block and the byte steps along y and z (0
// where the neighbour is not read), and the profile.
template <typename T> struct RowSlab {
    bool in, act;
    size_t row, dj, dk;
    T s, c, d;
};
template <typename T> using RowLineC = const __attribute__((address_space(4))) RowLine<T> *;
template <typename T> __device__ __forceinline__ RowLine<T> row_line(gptr<const RowLine<T>> l, int n)
{
    RowLineC<T> p = (RowLineC<T>)l.p + n;
    return {p->has, p->act, p->off, p->ks, p->s, p->c, p->d, p->m, p->t};
}
template <typename T> __device__ __forceinline__ RowSlab<T> row_slab_y(const RowLine<T> &l, int nx, int k)
{
    return {l.has != 0, l.act != 0, (size_t)((long long)l.off + (long long)l.ks * k) * sizeof(T),
            l.act ? (size_t)nx * sizeof(T) : 0, (size_t)l.ks * sizeof(T), l.s, l.c, l.d};
}
template <typename T> __device__ __forceinline__ RowSlab<T> row_slab_z(const RowLine<T> &l, int nx, int ny, int j)
{
    return {l.has != 0, l.act != 0, (size_t)((long long)l.off + (long long)nx * j) * sizeof(T), (size_t)nx * sizeof(T),
            l.act ? (size_t)nx * ny * sizeof(T) : 0, l.s, l.c, l.d};
}
// The x layer of a lane's node i on row (j, k): the lane's slab is an offset in the axis's
// block.  Lanes outside read element 0.
struct RowX {
    bool own, act;
    unsigned o, di, dj, dk;
};
template <typename T> __device__ __forceinline__ RowX row_x(const RowGeo &g, int i, int j, int k)
{
    RowX x;
    const bool lo = i < g.xa, hi = i >= g.xb && i < g.nx;
    const int n = lo ? g.n0 : g.n1;
    x.own = lo || hi;
    x.act = i < g.xi1 || (i >= g.xi2 && i < g.nx);
    const unsigned e = (unsigned)(lo ? i : g.d2 + i) + (unsigned)n * ((unsigned)j + (unsigned)g.ny * (unsigned)k);
    x.o = x.own ? e * (unsigned)sizeof(T) : 0u;
    x.di = x.act ? (unsigned)sizeof(T) : 0u;
    x.dj = x.own ? (unsigned)n * (unsigned)sizeof(T) : 0u;
    x.dk = x.own ? (unsigned)n * (unsigned)g.ny * (unsigned)sizeof(T) : 0u;
    return x;
}
// Whether a wavefront's points i0 .. i0 + 63 can meet an x slab.
__device__ __forceinline__ bool row_meets_x(const RowGeo &g, int i0) { return i0 < g.xa || i0 + RX > g.xb; }

// Layer auxiliaries one point's terms read: for the pressure the point and its forward
// neighbours, for the velocities the point and the pressure's backward neighbours.
template <typename T> struct QP { T u0, ui, uk, v0, vj, vk, w0, wk, p0; };
template <typename T> struct QV { T u0, v0, w0, p0, pi, pj, pk; };

// Layer coefficients of one axis at the point.
template <typename T> struct Lay { T s, c, d; bool act; };

// The layer terms of the pressure increment (air.cpp:2044-2292), x, y, z slabs with their corner
// cross terms, in the reference's order (dp_layers' expressions on values).
template <typename T, bool TERRAIN, bool X, bool Y, bool Z>
__device__ __forceinline__ T row_dp_layers(const AirArgs<T> &a, const Nb<T> &n, const Lay<T> &lx, const Lay<T> &ly,
                                           const Lay<T> &lz, const QP<T> &x, const QP<T> &y, const QP<T> &z, T pc, T ddx,
                                           T ddy, T dwz, T r)
{
    const T dxi = a.g.dxi, dyi = a.g.dyi, dzi = a.g.dzi, dt = a.g.dt, gP = a.gP;
    const T mX = n.mX, mY = n.mY, mZ = n.mZ, zX = n.zX, zY = n.zY;
    auto fX = [&](const QP<T> &q) {
        T v = (mX * (q.ui - q.u0)) * dxi;
        if constexpr (TERRAIN) v = v + (zX * (q.uk - q.u0)) * dzi;
        return v;
    };
    auto fY = [&](const QP<T> &q) {
        T v = (mY * (q.vj - q.v0)) * dyi;
        if constexpr (TERRAIN) v = v + (zY * (q.vk - q.v0)) * dzi;
        return v;
    };
    if constexpr (X) {
        const T A = (lx.c * (gP * ddx)) * dt;
        const T B = (lx.s * (pc + gP * (fY(x) + ((mZ * (x.wk - x.w0)) * dzi)))) * dt;
        const T s = r + (A - B);
        r = lx.act ? s : r;
    }
    if constexpr (Y) {
        const T A = (ly.c * (gP * ddy)) * dt;
        const T B = (ly.s * (pc + gP * (fX(y) + ((mZ * (y.wk - y.w0)) * dzi)))) * dt;
        T s = r + (A - B);
        if constexpr (X) {
            const T t1 = (lx.d * ly.s) * fX(x);
            const T t2 = (ly.d * lx.s) * fY(x);
            const T c = s + (-((x.p0 * lx.s) * ly.s + gP * (t1 + t2))) * dt;
            s = lx.act ? c : s;
        }
        r = ly.act ? s : r;
    }
    if constexpr (Z) {
        const T A = (((lz.c * a.gam) * a.Pav) * ((mZ * dwz) * dzi)) * dt;
        T inner;
        if constexpr (TERRAIN) {
            inner = (((((mX * (z.ui - z.u0)) * dxi) + ((zX * (z.uk - z.u0)) * dzi)) + ((mY * (z.vj - z.v0)) * dyi)) +
                     ((zY * (z.vk - z.v0)) * dzi));
        } else {
            inner = ((mX * (z.ui - z.u0)) * dxi) + ((mY * (z.vj - z.v0)) * dyi);
        }
        const T B = (lz.s * (pc + gP * inner)) * dt;
        T s = r + (A - B);
        if constexpr (X) {
            const T t1 = (lx.d * lz.s) * fX(x);
            const T t2 = (lz.d * lx.s) * ((mZ * (x.wk - x.w0)) * dzi);
            const T c = s + (-((x.p0 * lx.s) * lz.s + gP * (t1 + t2))) * dt;
            s = lx.act ? c : s;
        }
        if constexpr (Y) {
            const T t1 = (ly.d * lz.s) * fY(y);
            const T t2 = (lz.d * ly.s) * ((mZ * (y.wk - y.w0)) * dzi);
            const T c = s + (-((y.p0 * ly.s) * lz.s + gP * (t1 + t2))) * dt;
            s = ly.act ? c : s;
        }
        r = lz.act ? s : r;
    }
    return r;
}

// The layer terms of the velocity increments (air.cpp:1579-1905), as duvw_layers on values.
template <typename T, bool TERRAIN, bool X, bool Y, bool Z>
__device__ __forceinline__ void row_duvw_layers(const AirArgs<T> &a, const Nb<T> &n, const Lay<T> &lx, const Lay<T> &ly,
                                                const Lay<T> &lz, const QV<T> &x, const QV<T> &y, const QV<T> &z, T uc, T vc,
                                                T wc, T gpx, T gpy, T gpz, T &du, T &dv, T &dw)
{
    const T dxi = a.g.dxi, dyi = a.g.dyi, dzi = a.g.dzi, dt = a.g.dt, Aav = a.Aav;
    const T mX = n.mX, mY = n.mY, mZ = n.mZ, zX = n.zX, zY = n.zY;
    auto bX = [&](const QV<T> &q) {
        T v = (mX * (q.p0 - q.pi)) * dxi;
        if constexpr (TERRAIN) v = v + (zX * (q.p0 - q.pk)) * dzi;
        return v;
    };
    auto bY = [&](const QV<T> &q) {
        T v = (mY * (q.p0 - q.pj)) * dyi;
        if constexpr (TERRAIN) v = v + (zY * (q.p0 - q.pk)) * dzi;
        return v;
    };
    auto bZ = [&](const QV<T> &q) { return (mZ * (q.p0 - q.pk)) * dzi; };
    if constexpr (X) {
        const T sx = lx.s;
        const T u = du + (((-sx) * uc) * dt + (lx.c * (Aav * gpx)) * dt);
        const T v = dv + ((-sx) * (vc + Aav * bY(x))) * dt;
        const T w = dw + ((-sx) * (wc + Aav * bZ(x))) * dt;
        du = lx.act ? u : du; dv = lx.act ? v : dv; dw = lx.act ? w : dw;
    }
    if constexpr (Y) {
        const T sy = ly.s;
        T u = du + ((-sy) * (uc + Aav * bX(y))) * dt;
        T v = dv + (((ly.c * Aav) * gpy) * dt - (sy * vc) * dt);
        T w = dw + ((-sy) * (wc + Aav * bZ(y))) * dt;
        if constexpr (X) {
            const T sx = lx.s;
            const T cu = u + (-((x.u0 * sx) * sy + ((lx.d * sy) * Aav) * bX(x))) * dt;
            const T cv = v + (-((x.v0 * sx) * sy + ((ly.d * sx) * Aav) * bY(x))) * dt;
            const T cw = w + (((-x.w0) * sx) * sy) * dt;
            u = lx.act ? cu : u; v = lx.act ? cv : v; w = lx.act ? cw : w;
        }
        du = ly.act ? u : du; dv = ly.act ? v : dv; dw = ly.act ? w : dw;
    }
    if constexpr (Z) {
        const T sz = lz.s;
        T u = du + ((-sz) * (uc + Aav * bX(z))) * dt;
        T v = dv + ((-sz) * (vc + Aav * bY(z))) * dt;
        T w = dw + (((lz.c * Aav) * gpz) * dt - (sz * wc) * dt);
        if constexpr (X) {
            const T sx = lx.s;
            const T cu = u + (-((x.u0 * sx) * sz + ((lx.d * sz) * Aav) * bX(x))) * dt;
            const T cv = v + (((-x.v0) * sx) * sz) * dt;
            const T cw = w + (-((x.w0 * sx) * sz + ((lz.d * sx) * Aav) * bZ(x))) * dt;
            u = lx.act ? cu : u; v = lx.act ? cv : v; w = lx.act ? cw : w;
        }
        if constexpr (Y) {
            const T sy = ly.s;
            const T cu = u + (((-y.u0) * sy) * sz) * dt;
            const T cv = v + (-((y.v0 * sy) * sz + ((ly.d * sz) * Aav) * bY(y))) * dt;
            const T cw = w + (-((y.w0 * sy) * sz + ((lz.d * sy) * Aav) * bZ(y))) * dt;
            u = ly.act ? cu : u; v = ly.act ? cv : v; w = ly.act ? cw : w;
        }
        du = lz.act ? u : du; dv = lz.act ? v : dv; dw = lz.act ? w : dw;
    }
}

// The column's part of the metric at point i of row j: x, and over terrain sh, hx, hy.
template <typename T> struct RowColumn { T x, sh, hx, hy; };
// op: the column's byte offset from row j's first point (of the lane's row, where that differs).
template <typename T, bool TERRAIN>
__device__ __forceinline__ RowColumn<T> row_column(const Grid<T> &g, int nx, int i, int j, unsigned op)
{
    const unsigned o = op;
    RowColumn<T> c{ldr<T>(g.mx, 0, (unsigned)i * (unsigned)sizeof(T)), T(0), T(0), T(0)};
    if constexpr (TERRAIN) {
        const size_t r = (size_t)nx * j * sizeof(T);
        c.sh = ldr<T>(g.tsh, r, o);
        c.hx = ldr<T>(g.thx, r, o);
        c.hy = ldr<T>(g.thy, r, o);
    }
    return c;
}
// Inverse metric from the column's, the row's and the plane's values: metric / metric_terrain.
template <typename T, bool TERRAIN> __device__ __forceinline__ void row_metric(const RowColumn<T> &c, T yy, T zk, T tk, Nb<T> &n)
{
    n.zX = T(0); n.zY = T(0);
    const T xx = c.x;
    if constexpr (TERRAIN) {
        const T zz = zk * c.sh;
        const T Zx = c.hx * tk, Zy = c.hy * tk;
        const T J = T(1) / (xx * yy * zz);
        n.mX = (yy * zz) * J;
        n.mY = (xx * zz) * J;
        n.mZ = (xx * yy) * J;
        n.zX = (-(yy * Zx)) * J;
        n.zY = (-(xx * Zy)) * J;
    } else if constexpr (std::is_same<T, double>::value) {
        const double J = 1.0 / (xx * yy * zk);
        n.mX = (yy * zk) * J;
        n.mY = (xx * zk) * J;
        n.mZ = (xx * yy) * J;
    } else {
        n.mX = xx; n.mY = yy; n.mZ = zk;
    }
}
template <typename T, bool TERRAIN>
__device__ __forceinline__ void row_metric(const Grid<T> &g, int nx, int i, int j, T yy, T zk, T tk, Nb<T> &n)
{
    row_metric<T, TERRAIN>(row_column<T, TERRAIN>(g, nx, i, j, (unsigned)i * (unsigned)sizeof(T)), yy, zk, tk, n);
}

// Reader of a field at offsets (di, dj, dk) from the lane's point.
template <typename T> struct RowAt {
    size_t row, snx, sxy;
    unsigned o;
    __device__ __forceinline__ T operator()(gptr<const T> f, int di, int dj, int dk) const
    {
        return ldr<T>(f, row + (ptrdiff_t)dj * (ptrdiff_t)snx + (ptrdiff_t)dk * (ptrdiff_t)sxy, o, di * (int)sizeof(T));
    }
};

// Reader of the state around a point: field C (0 .. 3: u v w p, 4: the pressure the velocities
// read, of level n+1 in the FB step) at an offset.
template <typename T> struct RowState {
    const Grid<T> &g;
    const RowAt<T> &at;
    template <int C> __device__ __forceinline__ T get(int di, int dj, int dk) const
    {
        return at(C == 0 ? g.un : C == 1 ? g.vn : C == 2 ? g.wn : C == 3 ? g.pn : g.pnn, di, dj, dk);
    }
};

// The pressure increment without the layer terms, with the damped terms they use: dp_core for
// no mean flow and the log wind (WM 0, 2), the three-component mean flow (WM 1) in the form of
// air_dp.  n holds the metric; CEN: central convective differences (RK4).  The state comes
// from st, the mean flow from at.
template <typename T, int WM, bool TERRAIN, bool CEN, typename W, typename S>
__device__ __forceinline__ T row_dp(const AirArgs<T> &a, const W &at, const S &st, Nb<T> &n, T &ddx, T &ddy, T &dwz)
{
    const Grid<T> &g = a.g;
    n.pc = st.template get<3>(0, 0, 0);
    n.uc = st.template get<0>(0, 0, 0); n.vc = st.template get<1>(0, 0, 0); n.wc = st.template get<2>(0, 0, 0);
    n.u_ip = st.template get<0>(1, 0, 0); n.v_jp = st.template get<1>(0, 1, 0); n.w_kp = st.template get<2>(0, 0, 1);
    if constexpr (TERRAIN) { n.u_kp = st.template get<0>(0, 0, 1); n.v_kp = st.template get<1>(0, 0, 1); }
    if constexpr (WM == 2) {
        n.Vc = at(a.V, 0, 0, 0); n.V_jp = at(a.V, 0, 1, 0); n.V_jm = at(a.V, 0, -1, 0);
        n.p_jm = st.template get<3>(0, -1, 0);
        if constexpr (CEN) n.p_jp = st.template get<3>(0, 1, 0);
        if constexpr (TERRAIN) {
            n.V_kp = at(a.V, 0, 0, 1); n.V_km = at(a.V, 0, 0, -1);
            n.p_km = st.template get<3>(0, 0, -1);
            if constexpr (CEN) n.p_kp = st.template get<3>(0, 0, 1);
        }
    }
    if constexpr (WM != 1) {
        return dp_core<T, WM, TERRAIN, CEN>(a, n, ddx, ddy, dwz);
    } else {
        const T r0 = dp_core<T, 0, TERRAIN, CEN>(a, n, ddx, ddy, dwz);  // (-gam Pav dt) div
        const T dxi = g.dxi, dyi = g.dyi, dzi = g.dzi, dt = g.dt;
        const T mX = n.mX, mY = n.mY, mZ = n.mZ, zX = n.zX, zY = n.zY, pc = n.pc;
        const T Uc = at(a.U, 0, 0, 0), Vc = at(a.V, 0, 0, 0), Wc = at(a.W, 0, 0, 0);
        const T c1 = ((Uc * mX) * dxi) * dt, c2 = ((Vc * mY) * dyi) * dt;
        T c3;
        T UX = ((mX * (at(a.U, 1, 0, 0) - at(a.U, -1, 0, 0))) * dxi) * T(0.5);
        T VY = ((mY * (at(a.V, 0, 1, 0) - at(a.V, 0, -1, 0))) * dyi) * T(0.5);
        const T WZ = ((mZ * (at(a.W, 0, 0, 1) - at(a.W, 0, 0, -1))) * dzi) * T(0.5);
        if constexpr (TERRAIN) {
            c3 = ((((Uc * zX) + (Vc * zY)) + (Wc * mZ)) * dzi) * dt;
            UX = UX + ((zX * (at(a.U, 0, 0, 1) - at(a.U, 0, 0, -1))) * dzi) * T(0.5);
            VY = VY + ((zY * (at(a.V, 0, 0, 1) - at(a.V, 0, 0, -1))) * dzi) * T(0.5);
        } else {
            c3 = ((Wc * mZ) * dzi) * dt;
        }
        T r;
        if constexpr (CEN)
            r = ((-c1) * ((st.template get<3>(1, 0, 0) - st.template get<3>(-1, 0, 0)) * T(0.5)) - c2 * ((st.template get<3>(0, 1, 0) - st.template get<3>(0, -1, 0)) * T(0.5))) -
                c3 * ((st.template get<3>(0, 0, 1) - st.template get<3>(0, 0, -1)) * T(0.5));
        else
            r = ((-c1) * (pc - st.template get<3>(-1, 0, 0)) - c2 * (pc - st.template get<3>(0, -1, 0))) - c3 * (pc - st.template get<3>(0, 0, -1));
        r += (((-a.gam) * pc) * dt) * ((UX + VY) + WZ);
        return r + r0;
    }
}

// The velocity increments without the layer terms, with the pressure gradients they use:
// duvw_core (WM 0, 2), or the form of air_duvw (WM 1).
template <typename T, int WM, bool TERRAIN, bool CEN, typename W, typename S>
__device__ __forceinline__ void row_duvw(const AirArgs<T> &a, const W &at, const S &st, Nb<T> &n, T &gpx, T &gpy, T &gpz, T &du,
                                         T &dv, T &dw)
{
    n.uc = st.template get<0>(0, 0, 0); n.vc = st.template get<1>(0, 0, 0); n.wc = st.template get<2>(0, 0, 0);
    n.pc = st.template get<4>(0, 0, 0);
    n.p_im = st.template get<4>(-1, 0, 0); n.p_jm = st.template get<4>(0, -1, 0); n.p_km = st.template get<4>(0, 0, -1);
    if constexpr (WM == 2) {
        n.Vc = at(a.V, 0, 0, 0);
        n.V_ip = at(a.V, 1, 0, 0); n.V_im = at(a.V, -1, 0, 0); n.V_jp = at(a.V, 0, 1, 0); n.V_jm = at(a.V, 0, -1, 0);
        n.V_kp = at(a.V, 0, 0, 1); n.V_km = at(a.V, 0, 0, -1);
        n.u_jp = st.template get<0>(0, 1, 0); n.v_jp = st.template get<1>(0, 1, 0); n.w_jp = st.template get<2>(0, 1, 0);
        if constexpr (CEN) { n.u_jm = st.template get<0>(0, -1, 0); n.v_jm = st.template get<1>(0, -1, 0); n.w_jm = st.template get<2>(0, -1, 0); }
        if constexpr (TERRAIN) {
            n.u_kp = st.template get<0>(0, 0, 1); n.v_kp = st.template get<1>(0, 0, 1); n.w_kp = st.template get<2>(0, 0, 1);
            if constexpr (CEN) { n.u_km = st.template get<0>(0, 0, -1); n.v_km = st.template get<1>(0, 0, -1); n.w_km = st.template get<2>(0, 0, -1); }
        }
    }
    if constexpr (WM != 1) {
        duvw_core<T, WM, TERRAIN, CEN>(a, n, gpx, gpy, gpz, du, dv, dw);
    } else {
        T d0, d1, d2;
        duvw_core<T, 0, TERRAIN, CEN>(a, n, gpx, gpy, gpz, d0, d1, d2);  // (-Aav dt) grad p
        const T dxi = a.g.dxi, dyi = a.g.dyi, dzi = a.g.dzi, dt = a.g.dt;
        const T mX = n.mX, mY = n.mY, mZ = n.mZ, zX = n.zX, zY = n.zY, uc = n.uc, vc = n.vc, wc = n.wc;
        const T Uc = at(a.U, 0, 0, 0), Vc = at(a.V, 0, 0, 0), Wc = at(a.W, 0, 0, 0);
        const T c1 = ((Uc * mX) * dxi) * dt, c2 = ((Vc * mY) * dyi) * dt;
        T c3;
        if constexpr (TERRAIN) c3 = ((((Uc * zX) + (Vc * zY)) + (Wc * mZ)) * dzi) * dt;
        else c3 = ((Wc * mZ) * dzi) * dt;
        auto gx = [&](gptr<const T> F) {
            T q = ((mX * (at(F, 1, 0, 0) - at(F, -1, 0, 0))) * dxi) * T(0.5);
            if constexpr (TERRAIN) q = q + ((zX * (at(F, 0, 0, 1) - at(F, 0, 0, -1))) * dzi) * T(0.5);
            return q;
        };
        auto gy = [&](gptr<const T> F) {
            T q = ((mY * (at(F, 0, 1, 0) - at(F, 0, -1, 0))) * dyi) * T(0.5);
            if constexpr (TERRAIN) q = q + ((zY * (at(F, 0, 0, 1) - at(F, 0, 0, -1))) * dzi) * T(0.5);
            return q;
        };
        auto gz = [&](gptr<const T> F) { return ((mZ * (at(F, 0, 0, 1) - at(F, 0, 0, -1))) * dzi) * T(0.5); };
        auto cv = [&](auto C, T fc) {
            constexpr int F = decltype(C)::value;
            if constexpr (CEN)
                return ((-c1) * ((st.template get<F>(1, 0, 0) - st.template get<F>(-1, 0, 0)) * T(0.5)) -
                        c2 * ((st.template get<F>(0, 1, 0) - st.template get<F>(0, -1, 0)) * T(0.5))) -
                       c3 * ((st.template get<F>(0, 0, 1) - st.template get<F>(0, 0, -1)) * T(0.5));
            else
                return ((-c1) * (st.template get<F>(1, 0, 0) - fc) - c2 * (st.template get<F>(0, 1, 0) - fc)) - c3 * (st.template get<F>(0, 0, 1) - fc);
        };
        du = cv(std::integral_constant<int, 0>{}, uc);
        du += (((-uc) * gx(a.U)) * dt - (vc * gy(a.U)) * dt) - (wc * gz(a.U)) * dt;
        du += d0;
        dv = cv(std::integral_constant<int, 1>{}, vc);
        dv += (((-uc) * gx(a.V)) * dt - (vc * gy(a.V)) * dt) - (wc * gz(a.V)) * dt;
        dv += d1;
        dw = cv(std::integral_constant<int, 2>{}, wc);
        dw += (((-uc) * gx(a.W)) * dt - (vc * gy(a.W)) * dt) - (wc * gz(a.W)) * dt;
        dw += d2;
    }
}

// Increment of a porous point (porous.cpp:77-95): dt div of the velocities and, for the
// velocities, the pressure gradient.
template <typename T, bool TERRAIN> __device__ __forceinline__ void row_pore_grad(const Grid<T> &g, const RowAt<T> &at, const Nb<T> &n,
                                                                                  gptr<const T> p, T &gx, T &gy, T &gz)
{
    const T pc = at(p, 0, 0, 0), bz = pc - at(p, 0, 0, -1);
    gx = (n.mX * (pc - at(p, -1, 0, 0))) * g.dxi;
    gy = (n.mY * (pc - at(p, 0, -1, 0))) * g.dyi;
    gz = (n.mZ * bz) * g.dzi;
    if constexpr (TERRAIN) {
        gx = gx + (n.zX * bz) * g.dzi;
        gy = gy + (n.zY * bz) * g.dzi;
    }
}

}  // namespace

}  // namespace lee
