// lee_fb.hip -- FB_p_v step in row form: one launch per phase over the air, the porous layer, the
// ground interface plane, every face and the receivers (two launches over a large grid, whose
// interior outside every layer runs a kernel without layer terms).
//
// The general form (lee_kernels.hip, lee_bc.hip) takes five launches for a phase's air points,
// one for the porous layer and one for the faces.  Here the wavefront that computes a row next
// to a face stores the face's row as well, so no launch waits for another inside a phase.  A face node's
// value is its interior neighbour's (calculation_2D.cpp:646-864), zero for the velocity normal to
// the face, or the three-row extrapolation of the East pressure, for which the last tile row
// exchanges its rows through LDS; air and porous layer copy each other's planes
// (calculation_2D.cpp:865-985) the same way.  The node order of the reference's face chain is
// that of the walks in lee_bc.hip: x faces over y faces over the top, the ground last.  A row's
// last tile of at most 21 columns runs as a strip, several rows a wavefront (141 x 201 x 441 FP64
// with the East TDBC, rows of 64 + 64 + 13: 604 -> 566 us a step).
#include "lee_faces.h"
#include "lee_row.h"

#include <algorithm>

namespace lee {

namespace {

enum { RK_AIR = 0, RK_PORE = 1, RK_GROUND = 2, RK_REC = 3 };

// Tile of a block: what it computes, its plane, its tile column and tile row.
struct RowTile {
    int kind, k, tx, ty;
    long long rec;  // first receiver of the block
    int strip;      // a strip's block (RowLaunch), or -1
};
template <bool RING> __device__ __forceinline__ RowTile row_tile(const RowLaunch &l)
{
    RowTile t;
    t.rec = 0;
    t.strip = -1;
    if constexpr (!RING) {
        const int z = blockIdx.z;
        t.tx = blockIdx.x; t.ty = blockIdx.y;
        t.kind = z < l.zair ? RK_AIR : z < l.zair + l.zpore ? RK_PORE : z < l.zair + l.zpore + l.zground ? RK_GROUND : RK_REC;
        t.k = t.kind == RK_AIR ? z + 1 : t.kind == RK_PORE ? z - l.zair + 1 : 0;
        if (t.kind == RK_REC)
            t.rec = ((long long)(z - l.zair - l.zpore - l.zground) * l.nty + t.ty) * l.ntx + t.tx;
    } else {
        const int b = blockIdx.x, full = l.ntx * l.nty;
        // sections: planes below the interior, above it, the ring around it, porous, ground, receivers
        int s = 0, f = 0, per = full, k0 = 1;
        if (b >= l.first[1]) { s = 1; f = l.first[1]; k0 = l.kb; }
        if (b >= l.first[2]) { s = 2; f = l.first[2]; k0 = l.ka; per = l.nring; }
        if (b >= l.first[3]) { s = 3; f = l.first[3]; k0 = 1; per = full; }
        if (b >= l.first[4]) { s = 4; f = l.first[4]; k0 = 0; }
        if (b >= l.first[5]) { s = 5; f = l.first[5]; }
        const int q = b - f, kk = q / per, idx = q - kk * per;
        t.kind = s <= 2 ? RK_AIR : s == 3 ? RK_PORE : s == 4 ? RK_GROUND : RK_REC;
        t.k = k0 + kk;
        t.rec = q;
        if (s == 2) {
            const int e = ((const __attribute__((address_space(4))) int *)l.ring)[idx];
            t.tx = e & 0xffff; t.ty = e >> 16;
            if (e & kStripBlock) t.strip = e & (kStripBlock - 1);
        } else {
            t.ty = idx / l.ntx;
            t.tx = idx - t.ty * l.ntx;
        }
    }
    return t;
}

// ---- pressure ---------------------------------------------------------------------------
// One air node of row (j, k) other than the lane's own: p and the Q_p of the slabs holding it.
template <typename T> __device__ __forceinline__ void node_p(const RowArgs<T> &A, const RowGeo &G, int i, int j, int k, T v)
{
    const AirArgs<T> &a = A.a;
    const unsigned o = (unsigned)i * (unsigned)sizeof(T);
    const RowSlab<T> y = row_slab_y(row_line(A.yl, j), G.nx, k), z = row_slab_z(row_line(A.zl, k), G.nx, G.ny, j);
    const RowX x = row_x<T>(G, i, j, k);
    const T q = a.g.dt * v;
    T ox = T(0), oy = T(0), oz = T(0);
    if (x.own) ox = ldr<T>(A.q[0].o[3], 0, x.o);
    if (y.in) oy = ldr<T>(A.q[1].o[3], y.row, o);
    if (z.in) oz = ldr<T>(A.q[2].o[3], z.row, o);
    str<T>(a.g.pnn, (size_t)G.nx * ((size_t)j + (size_t)G.ny * k) * sizeof(T), o, v);
    if (x.own) str<T>(A.q[0].n[3], 0, x.o, ox + q);
    if (y.in) str<T>(A.q[1].n[3], y.row, o, oy + q);
    if (z.in) str<T>(A.q[2].n[3], z.row, o, oz + q);
}
template <typename T> __device__ __forceinline__ void store_node(const Grid<T> &g, gptr<T> f, int i, int j, int k, T v)
{
    str<T>(f, (size_t)g.nx * ((size_t)j + (size_t)g.ny * k) * sizeof(T), (unsigned)i * (unsigned)sizeof(T), v);
}

// p^{n+1} of the lane's point, and the old Q_p of the lane's node in its x, y and z slabs.
template <typename T, int WM, bool TERRAIN, bool X, bool Y, bool Z>
__device__ __forceinline__ T fb_p_point(const RowArgs<T> &A, const RowGeo &G, const RowLane &l, const RowPos &ps, int k, const RowLine<T> &yl,
                                        const RowLine<T> &zl, const RowSlab<T> &sy, const RowSlab<T> &sz, const RowX &xn, T &qx,
                                        T &qy, T &qz)
{
    const AirArgs<T> &a = A.a;
    const Grid<T> &g = a.g;
    const size_t snx = (size_t)G.nx * sizeof(T), sxy = snx * G.ny;
    const unsigned op = ps.op, on = l.live ? ps.on : op, ox = (unsigned)l.ip * (unsigned)sizeof(T);
    const RowAt<T> at{snx * ps.jb + sxy * k, snx, sxy, op};
    Nb<T> n;
    row_metric<T, TERRAIN>(row_column<T, TERRAIN>(g, G.nx, l.ip, ps.jb, op), yl.m, zl.m, zl.t, n);
    Lay<T> lx{}, ly{}, lz{};
    QP<T> x{}, y{}, z{};
    if constexpr (X) {
        const RowX q = row_x<T>(G, l.ip, ps.j, k);
        lx = {ldr<T>(A.xs, 0, ox), ldr<T>(A.xc, 0, ox), (Y || Z) ? ldr<T>(A.xd, 0, ox) : T(0), q.act};
        const RowQ<T> &Q = A.q[0];
        x.v0 = ldr<T>(Q.o[1], 0, q.o); x.vj = ldr<T>(Q.o[1], 0, q.o + q.dj);
        x.w0 = ldr<T>(Q.o[2], 0, q.o); x.wk = ldr<T>(Q.o[2], 0, q.o + q.dk);
        if constexpr (TERRAIN) x.vk = ldr<T>(Q.o[1], 0, q.o + q.dk);
        if constexpr (Y || Z) {
            x.u0 = ldr<T>(Q.o[0], 0, q.o); x.ui = ldr<T>(Q.o[0], 0, q.o + q.di);
            if constexpr (TERRAIN) x.uk = ldr<T>(Q.o[0], 0, q.o + q.dk);
            x.p0 = ldr<T>(Q.o[3], 0, q.o);
        }
        qx = ldr<T>(Q.o[3], 0, xn.o);
    }
    if constexpr (Y) {
        ly = {sy.s, sy.c, sy.d, sy.act};
        const RowQ<T> &Q = A.q[1];
        y.u0 = ldr<T>(Q.o[0], sy.row, op); y.ui = ldr<T>(Q.o[0], sy.row, op, sizeof(T));
        y.w0 = ldr<T>(Q.o[2], sy.row, op); y.wk = ldr<T>(Q.o[2], sy.row + sy.dk, op);
        if constexpr (TERRAIN) y.uk = ldr<T>(Q.o[0], sy.row + sy.dk, op);
        if constexpr (Z) {
            y.v0 = ldr<T>(Q.o[1], sy.row, op); y.vj = ldr<T>(Q.o[1], sy.row + sy.dj, op);
            if constexpr (TERRAIN) y.vk = ldr<T>(Q.o[1], sy.row + sy.dk, op);
            y.p0 = ldr<T>(Q.o[3], sy.row, op);
        }
        qy = ldr<T>(Q.o[3], sy.row, on);
    }
    if constexpr (Z) {
        lz = {sz.s, sz.c, sz.d, sz.act};
        const RowQ<T> &Q = A.q[2];
        z.u0 = ldr<T>(Q.o[0], sz.row, op); z.ui = ldr<T>(Q.o[0], sz.row, op, sizeof(T));
        z.v0 = ldr<T>(Q.o[1], sz.row, op); z.vj = ldr<T>(Q.o[1], sz.row + sz.dj, op);
        if constexpr (TERRAIN) {
            z.uk = ldr<T>(Q.o[0], sz.row + sz.dk, op);
            z.vk = ldr<T>(Q.o[1], sz.row + sz.dk, op);
        }
        qz = ldr<T>(Q.o[3], sz.row, on);
    }
    T ddx, ddy, dwz;
    T r = row_dp<T, WM, TERRAIN, false>(a, at, RowState<T>{g, at}, n, ddx, ddy, dwz);
    r = row_dp_layers<T, TERRAIN, X, Y, Z>(a, n, lx, ly, lz, x, y, z, n.pc, ddx, ddy, dwz, r);
    return n.pc + r;
}

// The air point of a lane: stencil, stores of its node.  YS: the row may lie in a y layer.
template <typename T, int WM, bool TERRAIN, bool YS>
__device__ __forceinline__ T fb_p_air(const RowArgs<T> &A, const RowGeo &G, const RowLane &l, const RowPos &ps, int k, const RowLine<T> &yl,
                                      const RowLine<T> &zl, bool mx)
{
    const Grid<T> &g = A.a.g;
    const RowSlab<T> sy = row_slab_y(yl, G.nx, k), sz = row_slab_z(zl, G.nx, G.ny, ps.jb);
    const RowX xn = row_x<T>(G, l.in, ps.j, k);
    T qx = T(0), qy = T(0), qz = T(0), p;
#define LEE_BODY(X, Y, Z) p = fb_p_point<T, WM, TERRAIN, X, Y, Z>(A, G, l, ps, k, yl, zl, sy, sz, xn, qx, qy, qz)
    if (!sz.in) {
        if (!YS || !sy.in) { if (mx) LEE_BODY(true, false, false); else LEE_BODY(false, false, false); }
        else { if (mx) LEE_BODY(true, YS, false); else LEE_BODY(false, YS, false); }
    } else {
        if (!YS || !sy.in) { if (mx) LEE_BODY(true, false, true); else LEE_BODY(false, false, true); }
        else { if (mx) LEE_BODY(true, YS, true); else LEE_BODY(false, YS, true); }
    }
#undef LEE_BODY
    if (l.live) {
        str<T>(g.pnn, (size_t)G.nx * ((size_t)ps.jb + (size_t)G.ny * k) * sizeof(T), ps.on, p);
        const T dq = g.dt * p;
        if (xn.own) str<T>(A.q[0].n[3], 0, xn.o, qx + dq);
        if (YS && sy.in) str<T>(A.q[1].n[3], sy.row, ps.on, qy + dq);
        if (sz.in) str<T>(A.q[2].n[3], sz.row, ps.on, qz + dq);
    }
    return p;
}
// A strip's block in either phase.
template <typename T> __device__ __forceinline__ bool fb_strip(const RowArgs<T> &A, const RowGeo &G, const RowLaunch &L, int strip, RowLane &l,
                                                               RowPos &ps, RowLine<T> &yl, bool &mx)
{
    const RowStrip &S = L.strip[0];  // (a row's narrow last tile: the only one)
    if (!row_strip<T>(S, L.ja, L.jb, strip, G.nx, l, ps)) return false;
    yl = RowLine<T>{};
    yl.m = ldr<T>(A.a.g.my, 0, (unsigned)ps.j * (unsigned)sizeof(T));
    mx = S.x0 < G.xa || S.x0 + S.n > G.xb;
    return true;
}

// p^{n+1} of a porous point (porous.cpp:77-95).
template <typename T, bool TERRAIN> __device__ __forceinline__ T pore_p_point(const RowArgs<T> &A, const RowLane &l, int j, int k)
{
    const Grid<T> &g = A.b.pore;
    const size_t snx = (size_t)g.nx * sizeof(T), sxy = snx * g.ny;
    const RowAt<T> at{snx * j + sxy * k, snx, sxy, (unsigned)l.ip * (unsigned)sizeof(T)};
    Nb<T> n;
    row_metric<T, TERRAIN>(g, g.nx, l.ip, j, lds_<T>(g.my, j), lds_<T>(g.mz, k), TERRAIN ? lds_<T>(g.ttk, k) : T(0), n);
    const T uc = at(g.un, 0, 0, 0), vc = at(g.vn, 0, 0, 0), wc = at(g.wn, 0, 0, 0);
    const T dux = at(g.un, 1, 0, 0) - uc, dvy = at(g.vn, 0, 1, 0) - vc, dwz = at(g.wn, 0, 0, 1) - wc;
    T div;
    if constexpr (TERRAIN) {
        const T duz = at(g.un, 0, 0, 1) - uc, dvz = at(g.vn, 0, 0, 1) - vc;
        div = ((((n.mX * g.dxi) * dux + (n.zX * g.dzi) * duz) + (n.mY * g.dyi) * dvy) + (n.zY * g.dzi) * dvz) +
              (n.mZ * g.dzi) * dwz;
    } else {
        div = ((n.mX * g.dxi) * dux + (n.mY * g.dyi) * dvy) + (n.mZ * g.dzi) * dwz;
    }
    return at(g.pn, 0, 0, 0) + (-A.pgama) * div;
}

template <typename T, int WM, bool TERRAIN, bool RING>
__global__ __launch_bounds__(RX * RY) void k_row_p(const RowArgs<T> *__restrict__ ap, RowLaunch L, double *__restrict__ rec_out)
{
    const RowArgs<T> &A = *ap;
    const RowGeo G = A.geo;
    const Grid<T> &g = A.a.g;
    const int nx = G.nx, ny = G.ny, nz = G.nz;
    const int lane = threadIdx.x, tj = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    const RowTile t = row_tile<RING>(L);
    if (t.kind == RK_REC) {
        // receivers sample time level n, which this step does not modify (airpore.cpp:573-580)
        const long long r = t.rec * (RX * RY) + tj * RX + lane;
        if (r < G.nrec) {
            const long long q = A.b.rec_idx[r];
            double v = q >= 0 ? (double)g.pn[q] : 0.0;
            if (fabs(v) < 1.0e-100) v = 0.0;
            rec_out[r] = v;
        }
        return;
    }
    if (RING && t.strip >= 0) {
        RowLane l;
        RowPos ps;
        RowLine<T> yl;
        bool mx;
        if (fb_strip(A, G, L, t.strip, l, ps, yl, mx)) fb_p_air<T, WM, TERRAIN, false>(A, G, l, ps, t.k, yl, row_line(A.zl, t.k), mx);
        return;
    }
    const int jr = G.j0 + RY * t.ty + tj, k = t.k;
    const bool row_live = jr >= 1;
    const int j = row_live ? jr : 1;
    const RowLane l = row_lane(G.i0 + t.tx * RX + lane, nx, row_live);
    __shared__ T rows[RY][RX];
    const bool last = t.ty == L.nty - 1;  // holds rows ny-4 .. ny-2 (uniform over the block)
    T p;
    if (t.kind == RK_AIR) {
        p = fb_p_air<T, WM, TERRAIN, true>(A, G, l, row_pos<T>(l, j), k, row_line(A.yl, j), row_line(A.zl, k), row_meets_x(G, G.i0 + t.tx * RX));
    } else if (t.kind == RK_PORE) {
        const Grid<T> &h = A.b.pore;
        // (the top plane of an uncoupled layer keeps what it holds)
        if (k == G.pnz - 1) p = h.pnn[gidx(h, l.ip, j, k)];
        else p = pore_p_point<T, TERRAIN>(A, l, j, k);
        if (l.live) store_node(h, h.pnn, l.in, j, k, p);
    } else {
        // the plane k = 0 of the ground impedance, or of air over an uncoupled porous layer
        p = G.ground ? ground_p(A.b, l.ip, j) : g.pnn[gidx(g, l.ip, j, 0)];
        if (l.live) node_p(A, G, l.in, j, k, p);
    }
    T pe = T(0);
    if (last) {
        rows[tj][lane] = p;
        __syncthreads();
        if (jr == ny - 2) pe = T(15.0 / 8.0) * p - T(5.0 / 4.0) * rows[tj - 1][lane] + T(3.0 / 8.0) * rows[tj - 2][lane];
    }
    if (!l.live) return;
    // the face rows next to this one: West, East, then the top or the ground plane of each
    const bool top = t.kind == RK_AIR && k == nz - 2, floor = t.kind == RK_AIR && k == 1 && !G.ground && (!G.porous || G.coupled);
    const bool pore_top = t.kind == RK_PORE && k == G.pnz - 2, pore_low = t.kind == RK_PORE && k == 1;
    if (jr != 1 && jr != ny - 2 && !top && !floor && !pore_top && !pore_low) return;
#pragma unroll 1
    for (int c = 0; c < 3; ++c) {
        if (c == 1 && jr != 1) continue;
        if (c == 2 && jr != ny - 2) continue;
        const int jn = c == 0 ? j : c == 1 ? 0 : ny - 1;
        const T v = c == 2 ? pe : p;
        if (t.kind == RK_PORE) {
            const Grid<T> &h = A.b.pore;
            if (c) store_node(h, h.pnn, l.in, jn, k, v);
            if (pore_low) store_node(h, h.pnn, l.in, jn, 0, v);
            if (pore_top && G.coupled) node_p(A, G, l.in, jn, 0, v);
        } else {
            if (c) node_p(A, G, l.in, jn, k, v);
            if (top) node_p(A, G, l.in, jn, nz - 1, v);
            if (floor) {
                if (G.porous) store_node(A.b.pore, A.b.pore.pnn, l.in, jn, G.pnz - 1, v);
                else node_p(A, G, l.in, jn, 0, v);
            }
        }
    }
}

// ---- velocities -------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void node_v(const RowArgs<T> &A, const RowGeo &G, int i, int j, int k, T u, T v, T w)
{
    const Grid<T> &g = A.a.g;
    const unsigned o = (unsigned)i * (unsigned)sizeof(T);
    const size_t row = (size_t)G.nx * ((size_t)j + (size_t)G.ny * k) * sizeof(T);
    const RowSlab<T> y = row_slab_y(row_line(A.yl, j), G.nx, k), z = row_slab_z(row_line(A.zl, k), G.nx, G.ny, j);
    const RowX x = row_x<T>(G, i, j, k);
    const T f[3] = {u, v, w};
    T qx[3], qy[3], qz[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (x.own) qx[c] = ldr<T>(A.q[0].o[c], 0, x.o);
        if (y.in) qy[c] = ldr<T>(A.q[1].o[c], y.row, o);
        if (z.in) qz[c] = ldr<T>(A.q[2].o[c], z.row, o);
    }
    str<T>(g.unn, row, o, u); str<T>(g.vnn, row, o, v); str<T>(g.wnn, row, o, w);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (x.own) str<T>(A.q[0].n[c], 0, x.o, qx[c] + g.dt * f[c]);
        if (y.in) str<T>(A.q[1].n[c], y.row, o, qy[c] + g.dt * f[c]);
        if (z.in) str<T>(A.q[2].n[c], z.row, o, qz[c] + g.dt * f[c]);
    }
}
template <typename T> __device__ __forceinline__ void pore_node_v(const Grid<T> &h, int i, int j, int k, T u, T v, T w)
{
    store_node(h, h.unn, i, j, k, u); store_node(h, h.vnn, i, j, k, v); store_node(h, h.wnn, i, j, k, w);
}

template <typename T, int WM, bool TERRAIN, bool X, bool Y, bool Z>
__device__ __forceinline__ void fb_v_point(const RowArgs<T> &A, const RowGeo &G, const RowLane &l, const RowPos &ps, int k,
                                           const RowLine<T> &yl, const RowLine<T> &zl, const RowSlab<T> &sy, const RowSlab<T> &sz,
                                           const RowX &xn, T (&out)[3], T (&qx)[3], T (&qy)[3], T (&qz)[3])
{
    const AirArgs<T> &a = A.a;
    const Grid<T> &g = a.g;
    const size_t snx = (size_t)G.nx * sizeof(T), sxy = snx * G.ny;
    const unsigned op = ps.op, on = l.live ? ps.on : op, ox = (unsigned)l.ip * (unsigned)sizeof(T);
    const RowAt<T> at{snx * ps.jb + sxy * k, snx, sxy, op};
    Nb<T> n;
    row_metric<T, TERRAIN>(row_column<T, TERRAIN>(g, G.nx, l.ip, ps.jb, op), yl.m, zl.m, zl.t, n);
    Lay<T> lx{}, ly{}, lz{};
    QV<T> x{}, y{}, z{};
    if constexpr (X) {
        const RowX q = row_x<T>(G, l.ip, ps.j, k);
        lx = {ldr<T>(A.xs, 0, ox), ldr<T>(A.xc, 0, ox), (Y || Z) ? ldr<T>(A.xd, 0, ox) : T(0), q.act};
        const RowQ<T> &Q = A.q[0];
        x.p0 = ldr<T>(Q.n[3], 0, q.o); x.pj = ldr<T>(Q.n[3], 0, q.o - q.dj); x.pk = ldr<T>(Q.n[3], 0, q.o - q.dk);
        if constexpr (Y || Z) {
            x.pi = ldr<T>(Q.n[3], 0, q.o - q.di);
            x.u0 = ldr<T>(Q.o[0], 0, q.o); x.v0 = ldr<T>(Q.o[1], 0, q.o); x.w0 = ldr<T>(Q.o[2], 0, q.o);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) qx[c] = ldr<T>(Q.o[c], 0, xn.o);
    }
    if constexpr (Y) {
        ly = {sy.s, sy.c, sy.d, sy.act};
        const RowQ<T> &Q = A.q[1];
        y.p0 = ldr<T>(Q.n[3], sy.row, op); y.pi = ldr<T>(Q.n[3], sy.row, op, -(int)sizeof(T));
        y.pk = ldr<T>(Q.n[3], sy.row - sy.dk, op);
        if constexpr (Z) {
            y.pj = ldr<T>(Q.n[3], sy.row - sy.dj, op);
            y.u0 = ldr<T>(Q.o[0], sy.row, op); y.v0 = ldr<T>(Q.o[1], sy.row, op); y.w0 = ldr<T>(Q.o[2], sy.row, op);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) qy[c] = ldr<T>(Q.o[c], sy.row, on);
    }
    if constexpr (Z) {
        lz = {sz.s, sz.c, sz.d, sz.act};
        const RowQ<T> &Q = A.q[2];
        z.p0 = ldr<T>(Q.n[3], sz.row, op); z.pi = ldr<T>(Q.n[3], sz.row, op, -(int)sizeof(T));
        z.pj = ldr<T>(Q.n[3], sz.row - sz.dj, op);
        if constexpr (TERRAIN) z.pk = ldr<T>(Q.n[3], sz.row - sz.dk, op);
#pragma unroll
        for (int c = 0; c < 3; ++c) qz[c] = ldr<T>(Q.o[c], sz.row, on);
    }
    T gpx, gpy, gpz, du, dv, dw;
    row_duvw<T, WM, TERRAIN, false>(a, at, RowState<T>{g, at}, n, gpx, gpy, gpz, du, dv, dw);
    row_duvw_layers<T, TERRAIN, X, Y, Z>(a, n, lx, ly, lz, x, y, z, n.uc, n.vc, n.wc, gpx, gpy, gpz, du, dv, dw);
    out[0] = n.uc + du; out[1] = n.vc + dv; out[2] = n.wc + dw;
}

// The air point of a lane: stencil, stores of its node.
template <typename T, int WM, bool TERRAIN, bool YS>
__device__ __forceinline__ void fb_v_air(const RowArgs<T> &A, const RowGeo &G, const RowLane &l, const RowPos &ps, int k,
                                         const RowLine<T> &yl, const RowLine<T> &zl, bool mx, T (&f)[3])
{
    const Grid<T> &g = A.a.g;
    const RowSlab<T> sy = row_slab_y(yl, G.nx, k), sz = row_slab_z(zl, G.nx, G.ny, ps.jb);
    const RowX xn = row_x<T>(G, l.in, ps.j, k);
    T qx[3], qy[3], qz[3];
#define LEE_BODY(X, Y, Z) fb_v_point<T, WM, TERRAIN, X, Y, Z>(A, G, l, ps, k, yl, zl, sy, sz, xn, f, qx, qy, qz)
    if (!sz.in) {
        if (!YS || !sy.in) { if (mx) LEE_BODY(true, false, false); else LEE_BODY(false, false, false); }
        else { if (mx) LEE_BODY(true, YS, false); else LEE_BODY(false, YS, false); }
    } else {
        if (!YS || !sy.in) { if (mx) LEE_BODY(true, false, true); else LEE_BODY(false, false, true); }
        else { if (mx) LEE_BODY(true, YS, true); else LEE_BODY(false, YS, true); }
    }
#undef LEE_BODY
    if (!l.live) return;
    if (l.face) f[0] = T(0);
    const unsigned o = ps.on;
    const size_t row = (size_t)G.nx * ((size_t)ps.jb + (size_t)G.ny * k) * sizeof(T);
    str<T>(g.unn, row, o, f[0]); str<T>(g.vnn, row, o, f[1]); str<T>(g.wnn, row, o, f[2]);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (xn.own) str<T>(A.q[0].n[c], 0, xn.o, qx[c] + g.dt * f[c]);
        if (YS && sy.in) str<T>(A.q[1].n[c], sy.row, o, qy[c] + g.dt * f[c]);
        if (sz.in) str<T>(A.q[2].n[c], sz.row, o, qz[c] + g.dt * f[c]);
    }
}

// Velocities of a porous point (porous.cpp:112-135).
template <typename T, bool TERRAIN>
__device__ __forceinline__ void pore_v_point(const RowArgs<T> &A, const RowLane &l, int j, int k, T (&out)[3])
{
    const Grid<T> &g = A.b.pore;
    const size_t snx = (size_t)g.nx * sizeof(T), sxy = snx * g.ny;
    const RowAt<T> at{snx * j + sxy * k, snx, sxy, (unsigned)l.ip * (unsigned)sizeof(T)};
    Nb<T> n;
    row_metric<T, TERRAIN>(g, g.nx, l.ip, j, lds_<T>(g.my, j), lds_<T>(g.mz, k), TERRAIN ? lds_<T>(g.ttk, k) : T(0), n);
    T gx, gy, gz;
    row_pore_grad<T, TERRAIN>(g, at, n, g.pnn, gx, gy, gz);
    const T f = ((T(-1.0) * A.pinvb) * g.dt) * A.peff;
    const T uc = at(g.un, 0, 0, 0), vc = at(g.vn, 0, 0, 0), wc = at(g.wn, 0, 0, 0);
    out[0] = uc + ((f * gx + uc * A.pinvb) - uc);
    out[1] = vc + ((f * gy + vc * A.pinvb) - vc);
    out[2] = wc + ((f * gz + wc * A.pinvb) - wc);
}

template <typename T, int WM, bool TERRAIN, bool RING>
__global__ __launch_bounds__(RX * RY) void k_row_v(const RowArgs<T> *__restrict__ ap, RowLaunch L)
{
    const RowArgs<T> &A = *ap;
    const RowGeo G = A.geo;
    const Grid<T> &g = A.a.g;
    const int nx = G.nx, ny = G.ny, nz = G.nz;
    const int lane = threadIdx.x, tj = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    const RowTile t = row_tile<RING>(L);
    if (RING && t.strip >= 0) {
        RowLane l;
        RowPos ps;
        RowLine<T> yl;
        bool mx;
        T f[3];
        if (fb_strip(A, G, L, t.strip, l, ps, yl, mx)) fb_v_air<T, WM, TERRAIN, false>(A, G, l, ps, t.k, yl, row_line(A.zl, t.k), mx, f);
        return;
    }
    const int jr = G.j0 + RY * t.ty + tj, k = t.k;
    if (jr < 1) return;
    const int j = jr;
    const RowLane l = row_lane(G.i0 + t.tx * RX + lane, nx, true);
    T f[3];
    if (t.kind == RK_AIR) {
        fb_v_air<T, WM, TERRAIN, true>(A, G, l, row_pos<T>(l, j), k, row_line(A.yl, j), row_line(A.zl, k), row_meets_x(G, G.i0 + t.tx * RX), f);
        if (!l.live) return;
    } else if (t.kind == RK_PORE) {
        const Grid<T> &h = A.b.pore;
        if (k == G.pnz - 1) {
            const size_t e = gidx(h, l.ip, j, k);
            f[0] = h.unn[e]; f[1] = h.vnn[e]; f[2] = h.wnn[e];
        } else {
            pore_v_point<T, TERRAIN>(A, l, j, k, f);
        }
        if (!l.live) return;
        if (l.face) f[0] = T(0);
        pore_node_v(A.b.pore, l.in, j, k, f[0], f[1], f[2]);
    } else if (!G.ground) {
        const size_t e = gidx(g, l.ip, j, 0);
        f[0] = g.unn[e]; f[1] = g.vnn[e]; f[2] = g.wnn[e];
        if (!l.live) return;
        if (l.face) f[0] = T(0);
        node_v(A, G, l.in, j, k, f[0], f[1], f[2]);
    } else {
        // the ground interface plane: its velocities, then the impedance's histories with the
        // velocity into the ground (calculation_2D.cpp:1012-1017), read once
        const BCArgs<T> &b = A.b;
        f[0] = ground_vel(b, 0, l.ip, j);
        f[1] = ground_vel(b, 1, l.ip, j);
        const size_t e = (size_t)l.ip + (size_t)nx * j, nn = (size_t)nx * ny;
        double P[8];
        double temp_psi = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (q < b.gK) { P[q] = b.gpsi_old[q * nn + e]; temp_psi += b.gdecay[q] * P[q]; }
        const double wd = ground_w_of(b, l.ip, j, temp_psi);
        f[2] = (T)wd;
        if (!l.live) return;
        if (l.face) f[0] = T(0);
        node_v(A, G, l.in, j, k, f[0], f[1], f[2]);
        const double vg = -wd;
        if (!l.face) {
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (q < b.gK) b.gpsi_new[q * nn + e] = b.gdecay[q] * P[q] + (b.ggain[q] * vg) * b.gtb;
        }
    }
    const bool top = t.kind == RK_AIR && k == nz - 2, floor = t.kind == RK_AIR && k == 1 && !G.ground && (!G.porous || G.coupled);
    const bool pore_top = t.kind == RK_PORE && k == G.pnz - 2, pore_low = t.kind == RK_PORE && k == 1;
    if (jr != 1 && jr != ny - 2 && !top && !floor && !pore_top && !pore_low) return;
    // East velocity of air plane kn: the TDBC's, from the final boundary pressure, or zero
    auto east_v = [&](int kn) { return G.tdbc ? (T)tdbc_v(A.b, l.ip, kn) : T(0); };
    // the air node of row jn, plane kn on the East face also advances the TDBC's histories
    auto histories = [&](int kn) {
        const BCArgs<T> &b = A.b;
        const double vt = tdbc_v(b, l.in, kn);
        const size_t e = ((size_t)l.in + (size_t)nx * kn) * 6;
#pragma unroll
        for (int q = 0; q < 6; ++q) b.psi_new[e + q] = b.decay[q] * b.psi_old[e + q] + (b.gain[q] * vt) * b.tb;
    };
#pragma unroll 1
    for (int c = 0; c < 3; ++c) {
        if (c == 1 && jr != 1) continue;
        if (c == 2 && jr != ny - 2) continue;
        const int jn = c == 0 ? j : c == 1 ? 0 : ny - 1;
        const T u = f[0], v = c == 0 ? f[1] : T(0), w = f[2];
        if (t.kind == RK_PORE) {
            const Grid<T> &h = A.b.pore;
            if (c) pore_node_v(h, l.in, jn, k, u, v, w);
            if (pore_low) pore_node_v(h, l.in, jn, 0, u, v, T(0));
            if (pore_top && G.coupled) {
                node_v(A, G, l.in, jn, 0, u, v, w);
                if (c == 2 && G.tdbc) histories(0);
            }
        } else {
            if (c) {
                node_v(A, G, l.in, jn, k, u, c == 2 ? east_v(k) : v, w);
                if (c == 2 && G.tdbc) histories(k);
            }
            if (top) {
                node_v(A, G, l.in, jn, nz - 1, u, c == 2 ? east_v(nz - 1) : v, T(0));
                if (c == 2 && G.tdbc) histories(nz - 1);
            }
            if (floor) {
                const T ve = c == 2 ? east_v(1) : v;
                if (G.porous) {
                    pore_node_v(A.b.pore, l.in, jn, G.pnz - 1, u, ve, w);
                } else {
                    node_v(A, G, l.in, jn, 0, u, ve, T(0));
                    if (c == 2 && G.tdbc) histories(0);
                }
            }
        }
    }
}

// ---- the interior outside every layer and away from every face ---------------------------
// One point per lane.
template <typename T, int WM, bool TERRAIN, bool PRESSURE>
__global__ __launch_bounds__(RX * RY) void k_row_in(const RowArgs<T> *__restrict__ ap, RowBox bx)
{
    const RowArgs<T> &A = *ap;
    const AirArgs<T> &a = A.a;
    const Grid<T> &g = a.g;
    const int tj = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    const int i = bx.i0 + (bx.tx + (int)blockIdx.x) * RX + (int)threadIdx.x, k = bx.k + (int)blockIdx.z;
    const int j = bx.j0 + RY * (bx.ty + (int)blockIdx.y) + tj;
    const size_t snx = (size_t)g.nx * sizeof(T), sxy = snx * g.ny;
    const RowAt<T> at{snx * j + sxy * k, snx, sxy, (unsigned)i * (unsigned)sizeof(T)};
    Nb<T> n;
    row_metric<T, TERRAIN>(g, g.nx, i, j, lds_<T>(g.my, j), lds_<T>(g.mz, k), TERRAIN ? lds_<T>(g.ttk, k) : T(0), n);
    if constexpr (PRESSURE) {
        T ddx, ddy, dwz;
        const T r = row_dp<T, WM, TERRAIN, false>(a, at, RowState<T>{g, at}, n, ddx, ddy, dwz);
        str<T>(g.pnn, at.row, at.o, n.pc + r);
    } else {
        T gpx, gpy, gpz, du, dv, dw;
        row_duvw<T, WM, TERRAIN, false>(a, at, RowState<T>{g, at}, n, gpx, gpy, gpz, du, dv, dw);
        str<T>(g.unn, at.row, at.o, n.uc + du); str<T>(g.vnn, at.row, at.o, n.vc + dv); str<T>(g.wnn, at.row, at.o, n.wc + dw);
    }
}

// P consecutive points of a row per lane (16-byte accesses), 64 / P lanes a row and a wavefront a
// 64 x 4 tile, without a mean flow: the i +- 1 neighbour at the vector's end is a load of its own.
// Rows start aligned to the vector (nx a multiple of P).  On the 512 x 256 x 128 grid (FP32, P = 4)
// the interior took 45.4 + 55.1 us one point per lane and 41.2 + 42.2 us in this form.  Over terrain
// the pressure reads u and v at k + 1 and the per-column tables as well and was slower so (603 against
// 545 us on 1024 x 512 x 160): one point per lane there, as in FP64 (1-5 % slower in vectors).
template <typename T, int P> using VecP = T __attribute__((ext_vector_type(P)));
template <typename T, int P> __device__ __forceinline__ VecP<T, P> ldv(gptr<const T> f, size_t q)
{
    return *(const __attribute__((address_space(1))) VecP<T, P> *)(f.p + q);
}
template <typename T, int P> __device__ __forceinline__ void stv(gptr<T> f, size_t q, const VecP<T, P> &v)
{
    *(__attribute__((address_space(1))) VecP<T, P> *)(f.p + q) = v;
}
template <typename T, bool TERRAIN, bool PRESSURE, int P>
__global__ __launch_bounds__(256) void k_row_in_vec(const RowArgs<T> *__restrict__ ap, RowBox bx, int ntiles)
{
    typedef VecP<T, P> V;
    const RowArgs<T> &A = *ap;
    const AirArgs<T> &a = A.a;
    const Grid<T> &g = a.g;
    const int t = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (t >= ntiles) return;
    const int per = bx.nbx * bx.nby, kk = t / per, c = t - kk * per, ty = c / bx.nbx, tx = c - ty * bx.nbx;
    constexpr int LR = RX / P;
    const int lane = (int)(threadIdx.x & 63), row = lane / LR;
    const int i = bx.i0 + (bx.tx + tx) * RX + (lane - row * LR) * P, j = bx.j0 + RY * (bx.ty + ty) + row, k = bx.k + kk;
    const size_t nx = (size_t)g.nx, sxy = nx * g.ny, id = (size_t)i + nx * ((size_t)j + (size_t)g.ny * k);
    const V uc = ldv<T, P>(g.un, id), vc = ldv<T, P>(g.vn, id), wc = ldv<T, P>(g.wn, id);
    if constexpr (PRESSURE) {
        static_assert(!TERRAIN, "separable grids only");
        const V pc = ldv<T, P>(g.pn, id), vjp = ldv<T, P>(g.vn, id + nx), wkp = ldv<T, P>(g.wn, id + sxy);
        const T ulast = g.un[id + P];
        V out;
#pragma unroll
        for (int e = 0; e < P; ++e) {
            Nb<T> n;
            n.zX = T(0); n.zY = T(0);
            metric(g, i + e, j, k, n.mX, n.mY, n.mZ);
            n.pc = pc[e]; n.uc = uc[e]; n.vc = vc[e]; n.wc = wc[e];
            n.u_ip = e + 1 < P ? uc[(e + 1) & (P - 1)] : ulast;
            n.v_jp = vjp[e]; n.w_kp = wkp[e];
            T ddx, ddy, dwz;
            out[e] = pc[e] + dp_core<T, 0, false, false>(a, n, ddx, ddy, dwz);
        }
        stv<T, P>(g.pnn, id, out);
    } else {
        const V pc = ldv<T, P>(g.pnn, id), pjm = ldv<T, P>(g.pnn, id - nx), pkm = ldv<T, P>(g.pnn, id - sxy);
        const T pfirst = g.pnn[id - 1];
        V uo, vo, wo;
#pragma unroll
        for (int e = 0; e < P; ++e) {
            Nb<T> n;
            n.zX = T(0); n.zY = T(0);
            if constexpr (TERRAIN) metric_terrain(g, i + e, j, k, n.mX, n.mY, n.mZ, n.zX, n.zY);
            else metric(g, i + e, j, k, n.mX, n.mY, n.mZ);
            n.uc = uc[e]; n.vc = vc[e]; n.wc = wc[e];
            n.pc = pc[e];
            n.p_im = e > 0 ? pc[(e + P - 1) & (P - 1)] : pfirst;
            n.p_jm = pjm[e]; n.p_km = pkm[e];
            T gpx, gpy, gpz, du, dv, dw;
            duvw_core<T, 0, TERRAIN, false>(a, n, gpx, gpy, gpz, du, dv, dw);
            uo[e] = uc[e] + du; vo[e] = vc[e] + dv; wo[e] = wc[e] + dw;
        }
        stv<T, P>(g.unn, id, uo); stv<T, P>(g.vnn, id, vo); stv<T, P>(g.wnn, id, wo);
    }
}
template <typename T, bool TERRAIN, bool PRESSURE> void launch_in_vec(const RowArgs<T> *ad, const RowBox &b, hipStream_t s)
{
    const int nt = b.nbx * b.nby * b.nk;
    if constexpr (sizeof(T) == 4)
        hipLaunchKernelGGL((k_row_in_vec<T, TERRAIN, PRESSURE, 4>), dim3((unsigned)((nt + 3) / 4)), dim3(256), 0, s, ad, b, nt);
}

}  // namespace

template <typename T> void launch_row_p(const RowArgs<T> *ad, const RowPlan &pl, bool wind, bool terrain, bool split,
                                        bool vec, double *rec, hipStream_t s)
{
    const dim3 blk(RX, RY), box((unsigned)pl.in.nbx, (unsigned)pl.in.nby, (unsigned)pl.in.nk);
#define LEE_RP(W, TER)                                                                                              \
    do {                                                                                                            \
        if (split) {                                                                                                \
            if (sizeof(T) == 4 && vec && !TER && !W) launch_in_vec<T, false, true>(ad, pl.in, s);                                     \
            else hipLaunchKernelGGL((k_row_in<T, W, TER, true>), box, blk, 0, s, ad, pl.in);                        \
            hipLaunchKernelGGL((k_row_p<T, W, TER, true>), dim3((unsigned)pl.p.first[6]), blk, 0, s, ad, pl.p, rec); \
        } else if (!pl.w[0].grid) {                                                                                 \
            hipLaunchKernelGGL((k_row_p<T, W, TER, true>), dim3((unsigned)pl.w[0].first[6]), blk, 0, s, ad, pl.w[0], rec); \
        } else {                                                                                                    \
            hipLaunchKernelGGL((k_row_p<T, W, TER, false>), dim3((unsigned)pl.p.ntx, (unsigned)pl.p.nty, (unsigned)pl.p.z), blk, \
                               0, s, ad, pl.p, rec);                                                                \
        }                                                                                                           \
    } while (0)
    if (terrain) { if (wind) LEE_RP(1, true); else LEE_RP(0, true); }
    else { if (wind) LEE_RP(1, false); else LEE_RP(0, false); }
#undef LEE_RP
}
template <typename T> void launch_row_v(const RowArgs<T> *ad, const RowPlan &pl, bool wind, bool terrain, bool split,
                                        bool vec, hipStream_t s)
{
    const dim3 blk(RX, RY), box((unsigned)pl.in.nbx, (unsigned)pl.in.nby, (unsigned)pl.in.nk);
#define LEE_RV(W, TER)                                                                                              \
    do {                                                                                                            \
        if (split) {                                                                                                \
            if (sizeof(T) == 4 && vec && !W) launch_in_vec<T, TER, false>(ad, pl.in, s);                                              \
            else hipLaunchKernelGGL((k_row_in<T, W, TER, false>), box, blk, 0, s, ad, pl.in);                       \
            hipLaunchKernelGGL((k_row_v<T, W, TER, true>), dim3((unsigned)pl.v.first[6]), blk, 0, s, ad, pl.v);     \
        } else if (!pl.w[1].grid) {                                                                                 \
            hipLaunchKernelGGL((k_row_v<T, W, TER, true>), dim3((unsigned)pl.w[1].first[6]), blk, 0, s, ad, pl.w[1]); \
        } else {                                                                                                    \
            hipLaunchKernelGGL((k_row_v<T, W, TER, false>), dim3((unsigned)pl.v.ntx, (unsigned)pl.v.nty, (unsigned)pl.v.z), blk, \
                               0, s, ad, pl.v);                                                                     \
        }                                                                                                           \
    } while (0)
    if (terrain) { if (wind) LEE_RV(1, true); else LEE_RV(0, true); }
    else { if (wind) LEE_RV(1, false); else LEE_RV(0, false); }
#undef LEE_RV
}

// Launch plan of a domain: tile counts and, over a grid with an interior (outside every layer and
// not next to a face; FB: whole tiles of it), that box and the ring of tiles around it.
void row_plan(RowPlan &pl, std::vector<int> &ring, const RowGeom &m)
{
    const int i0 = row_left(m.nx), j0 = row_first(m.ny), ntx = (m.nx - i0 + RX - 1) / RX, nty = row_tiles(m.ny);
    // first and one-past-last point of the interior along each axis
    auto span = [](int n, const int *qn, const int *qlo, int w1, int w2, int &a, int &b) {
        a = 2; b = n - 2;
        if (qn[0]) a = std::max(a, qlo[0] + qn[0]);
        if (qn[1]) b = std::min(b, qlo[1]);
        a = std::max(a, w1);
        b = std::min(b, n - w2);
    };
    int xa, xb, ya, yb, za, zb;
    span(m.nx, m.qn, m.qlo, m.w[0], m.w[1], xa, xb);
    span(m.ny, m.qn + 2, m.qlo + 2, m.w[2], m.w[3], ya, yb);
    span(m.nz, m.qn + 4, m.qlo + 4, m.w[4], m.w[5], za, zb);
    const int tx0 = (xa - i0 + RX - 1) / RX, tx1 = (xb - i0) / RX;
    const int ty0 = (ya - j0 + RY - 1) / RY, ty1 = (yb - j0) / RY;
    pl = RowPlan{};
    pl.i0 = i0;
    pl.j0 = j0;
    pl.has_in = tx1 > tx0 && ty1 > ty0 && zb > za;
    if (pl.has_in) pl.in = RowBox{tx0, tx1 - tx0, ty0, ty1 - ty0, za, zb - za, i0, j0};
    if (m.rk4) {
        // any points, except the rows of the last tile row (it extrapolates the East pressure);
        // two tiles wide at least, so that no tile meets both ends
        RowPair &b = pl.pair;
        b.xa = xa; b.xb = xb; b.ya = ya; b.yb = std::min(yb, j0 + RY * (nty - 1)); b.za = za; b.zb = zb;
        const int wx = b.xb - b.xa, wy = b.yb - b.ya, wz = b.zb - b.za;
        pl.has_in = wx >= 2 * RX && wy >= 16 && wz >= 8;
        if (pl.has_in) {
            auto cut = [](int n, int most, int &parts, int &width) {
                parts = (n + most - 1) / most;
                width = (n + parts - 1) / parts;
                parts = (n + width - 1) / width;
            };
            cut(wx, RX - 2, b.nbx, b.wx);
            cut(wy, pair_rows(m.esz) - 2, b.nby, b.wy);
            // planes per block: one block a CU at a time, each with two planes more than its own
            const int cols = b.nbx * b.nby;
            long long best = -1;
            for (int nz = 1; nz <= 16 && nz * 4 <= wz; ++nz) {
                const int w = (wz + nz - 1) / nz;
                const long long cost = (long long)((cols * nz + 255) / 256) * (w + 2);
                if (best < 0 || cost < best) { best = cost; b.wz = w; b.nbz = (wz + w - 1) / w; }
            }
        }
    }
    const int full = ntx * nty, nrp = (m.nrec + full * RX * RY - 1) / (full * RX * RY);
    // tile rows outside the y layers, neither the first (face row) nor the last (East extrapolation)
    const int jy0 = m.qn[2] ? m.qlo[2] + m.qn[2] : 0, jy1 = m.qn[3] ? m.qlo[3] : m.ny;
    auto packs = [&](RowLaunch &l, int most, int xlo, int xhi, int ya, int yb) {  // strips [0, xlo) and [xhi, nx)
        const int ta = std::max(1, (std::max(ya, jy0) - j0 + RY - 1) / RY), tb = std::min(nty - 1, (std::min(yb, jy1) - j0) / RY);
        if (tb <= ta) return;
        for (int q = 0; q < 2; ++q) {
            const int x0 = q ? xhi : 0, n = q ? m.nx - xhi : xlo;
            if (n >= 1 && n <= most) l.strip[l.nstrip++] = RowStrip{x0, n, RX / n, 65536 / n + 1};
        }
        l.ja = j0 + RY * ta; l.jb = j0 + RY * tb;
    };
    auto packed = [&](const RowLaunch &l, int tx, int ty) {  // the tile's points are strips' (or the interior's)
        if (!l.nstrip || j0 + RY * ty < l.ja || j0 + RY * (ty + 1) > l.jb) return false;
        const int x0 = i0 + RX * tx, x1 = std::min(x0 + RX, m.nx);
        for (int q = 0; q < l.nstrip; ++q) {
            const int a = l.strip[q].x0, b = a + l.strip[q].n;
            if (std::max(a, x0) < std::min(b, x1)) return true;
        }
        return false;
    };
    for (int ph = 0; ph < 2; ++ph) {
        RowLaunch &l = ph ? pl.v : pl.p;
        l.ntx = ntx; l.nty = nty;
        l.zair = m.nz - 2;
        // an uncoupled porous layer: its top plane and the air's plane 0 are planes of their own
        l.zpore = m.pnz > 0 ? m.pnz - 2 + (m.coupled ? 0 : 1) : 0;
        l.zground = m.ground || (m.pnz > 0 && !m.coupled) ? 1 : 0;
        l.z = l.zair + l.zpore + l.zground + (ph ? 0 : nrp);
        l.ka = za; l.kb = zb;
        l.xa = pl.pair.xa; l.xb = pl.pair.xb; l.ya = pl.pair.ya; l.yb = pl.pair.yb;
        RowLaunch &w = pl.w[ph];
        {
            w = l;
            w.xa = w.xb = w.ya = w.yb = 0;
            w.ka = 2; w.kb = std::max(2, m.nz - 2);
            const int tail = i0 + RX * (ntx - 1);
            packs(w, RX / 3, 0, ntx > 1 ? tail : m.nx, 0, m.ny);
            w.grid = !w.nstrip;
            if (w.grid) w.ka = w.kb = 1;  // (an ensemble's blocks: whole planes)
            if (m.rk4 && pl.has_in) packs(l, RX / 2, l.xa, l.xb, l.ya, l.yb);
        }
        auto sections = [&](RowLaunch &r, int tiles) {
            r.nring = tiles ? tiles : 1;
            auto inverse = [](int d) { return d > 1 ? (unsigned)(((1ULL << 32) + d - 1) / d) : ~0u; };
            r.by_full = inverse(full); r.by_ntx = inverse(ntx); r.by_ring = inverse(r.nring);
            const int per[6] = {full * (r.ka - 1), full * (m.nz - 1 - r.kb), tiles * (r.kb - r.ka), full * r.zpore, full * r.zground,
                                ph ? 0 : (m.nrec + RX * RY - 1) / (RX * RY)};
            r.first[0] = 0;
            for (int q = 0; q < 6; ++q) r.first[q + 1] = r.first[q] + per[q];
        };
        if (!ph) {
            ring.clear();
            pl.list.clear();
            auto strips = [&](std::vector<int> &list, const RowLaunch &r, int ty) {  // those that start in tile row ty
                for (int q = 0; q < r.nstrip; ++q)
                    for (int b = 0; r.ja + RY * r.strip[q].rows * b < r.jb; ++b)
                        if ((r.ja + RY * r.strip[q].rows * b - j0) / RY == ty) list.push_back(kStripBlock | q << 20 | b);
            };
            for (int ty = 0; ty < nty; ++ty) {
                for (int tx = 0; tx < ntx; ++tx) {
                    const int e = tx | (ty << 16);
                    const bool in = m.rk4 ? i0 + RX * tx >= pl.pair.xa && i0 + RX * (tx + 1) <= pl.pair.xb &&
                                                j0 + RY * ty >= pl.pair.ya && j0 + RY * (ty + 1) <= pl.pair.yb
                                          : tx >= tx0 && tx < tx1 && ty >= ty0 && ty < ty1;
                    if (pl.has_in && !in && !packed(l, tx, ty)) ring.push_back(e);
                    if (!packed(w, tx, ty)) pl.list.push_back(e);
                }
                if (pl.has_in) strips(ring, l, ty);
                strips(pl.list, w, ty);
            }
        }
        if (pl.has_in) sections(l, (int)ring.size());
        else l.nring = 1;
        sections(w, (int)pl.list.size());
    }
}

#define LEE_INST(T)                                                                                                     \
    template void launch_row_p<T>(const RowArgs<T> *, const RowPlan &, bool, bool, bool, bool, double *, hipStream_t);      \
    template void launch_row_v<T>(const RowArgs<T> *, const RowPlan &, bool, bool, bool, bool, hipStream_t);
LEE_INST(double)
LEE_INST(float)
#undef LEE_INST

}  // namespace lee
