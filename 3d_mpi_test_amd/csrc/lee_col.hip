// lee_col.hip -- several FB_p_v steps per launch for narrow columns: a plane of at most 64 nodes
// and no layer but those along z (the learned ground's reflection columns: 6 x 6 x 640).
//
// By launches per phase such a step is bound by its two launches and by the dependent loads in
// each (arguments, row records, fields, face rows): 5-6 us a phase for 24 k points.  Here a
// workgroup holds a window of whole planes in LDS, one node per lane, and advances it nsteps
// steps; a step moves information by one plane, so the window carries `halo` planes on either
// side of the `own` planes whose nodes it stores, computed by the neighbours as well (each step
// only those that the owned ones still depend on), and nothing passes between workgroups.
// Level n is read from one set of buffers and level n + nsteps written to the other, the roles a
// single step alternates.  The porous layer's planes and the air's follow one another in the
// window; the two pairs of planes that copy each other across the interface (air 0 = porous
// top - 1, porous top = air 1) make a crossing two planes longer, a face that copies its
// neighbour one: halo >= nsteps + 3.  Planes past that range hold values that nothing reads.
//
// A face node computes its interior neighbour's point and takes over the value, as in lee_fb.hip;
// fields alternate between two LDS copies so that it still finds the old value.  The East
// pressure is read by nothing inside a step and follows in the velocity phase.  The arithmetic is
// the row form's (lee_core.h, lee_row.h): the same bits.
//
// 6 x 6 x 640 over 12 porous planes, FP64, us a step: 10.8 by launches per phase, 2.3 here (nine
// steps a launch: 7 us of launch and dependent loads, 1.5 us a step bound by the latency of
// LDS, the arithmetic chain and two barriers).  Computing the whole window in each step took
// 2.5, the coefficients held in scalar registers (46 spilled to vector lanes) the same 2.3.
#include "lee_faces.h"
#include "lee_row.h"

namespace lee {

namespace {

constexpr int CN = 1024;  // nodes of a window, one per lane

template <typename T>
__global__ __launch_bounds__(CN) void k_col(const RowArgs<T> *__restrict__ ap, int own, int halo, int nsteps, double *__restrict__ rec_out)
{
    __shared__ T F[2][4][CN];       // u v w p at the level read and the level written
    __shared__ T Q[4][CN];          // z layers' auxiliaries
    __shared__ double psi[2][8][kColPlane];  // ground impedance histories
    const RowArgs<T> &A = *ap;
    const RowGeo G = A.geo;
    const AirArgs<T> &a = A.a;
    const BCArgs<T> &b = A.b;
    const Grid<T> &g = a.g, &h = b.pore;
    const int nx = G.nx, ny = G.ny, nz = G.nz, pnz = G.porous ? G.pnz : 0, P = nx * ny, C = pnz + nz;
    const int c0 = (int)blockIdx.x * own, c1 = min(C, c0 + own), lo = max(0, c0 - halo), hi = min(C, c1 + halo);
    // the lane's node and the point it computes: the nearest interior one, in the plane a
    // horizontal face or the interface copies from (the node itself where that lies outside the window)
    const int e = threadIdx.x, cl = e / P, nd = e - cl * P, j = nd / nx, i = nd - j * nx, c = lo + cl;
    const bool live = c < hi, mine = live && c >= c0 && c < c1;
    const bool air = c >= pnz;
    const int k = air ? c - pnz : c;
    const int ip = min(max(i, 1), nx - 2), jp = min(max(j, 1), ny - 2);
    int cs = c;
    if (air) {
        if (k == nz - 1) cs = c - 1;
        if (k == 0 && !G.ground) cs = pnz ? c - 2 : c + 1;
    } else {
        if (k == 0) cs = c + 1;
        if (k == pnz - 1) cs = c + 2;
    }
    if (cs < lo || cs >= hi) cs = c;
    const bool sair = cs >= pnz;
    const int ks = sair ? cs - pnz : cs;
    const bool sground = sair && ks == 0 && G.ground;
    const int es = (cs - lo) * P + jp * nx + ip, up = es + (cs + 1 < hi ? P : 0), dn = es - (cs > lo ? P : 0);
    const bool xface = i == 0 || i == nx - 1, west = j == 0, east = j == ny - 1, inner = !xface && !west && !east;
    const bool rigid = air ? k == nz - 1 || (k == 0 && !G.ground && !pnz) : k == 0;  // w = 0
    Nb<T> n;
    Lay<T> lz{};
    bool lay = false, has = false;
    size_t qe = 0;
    const size_t ge = (size_t)nd + (size_t)P * k;
    n.zX = n.zY = T(0);
    n.mX = n.mY = n.mZ = T(0);
    if (live) {
        if (sground) {
            n.mX = (T)b.gmx[ip]; n.mY = (T)b.gmy[jp]; n.mZ = (T)b.gmz;
        } else if (sair) {
            metric(g, ip, jp, ks, n.mX, n.mY, n.mZ);
        } else {
            metric(h, ip, jp, ks, n.mX, n.mY, n.mZ);
        }
        if (sair) {
            const RowLine<T> l = A.zl.p[ks];
            lay = l.has;
            lz = {l.s, l.c, l.d, l.act != 0};
        }
        const Grid<T> &s = air ? g : h;
        F[0][0][e] = s.un[ge]; F[0][1][e] = s.vn[ge]; F[0][2][e] = s.wn[ge]; F[0][3][e] = s.pn[ge];
        if (air) {
            const RowLine<T> l = A.zl.p[k];
            has = l.has;
            qe = (size_t)l.off + (size_t)nd;
            if (has)
#pragma unroll
                for (int f = 0; f < 4; ++f) Q[f][e] = A.q[2].o[f][qe];
            if (G.ground && k == 0)
                for (int q = 0; q < b.gK; ++q) psi[0][q][nd] = b.gpsi_old[(size_t)q * P + nd];
        }
    }
    // receivers: the block that owns the plane, or the first for one outside the grid; a sample
    // is the pressure of level n (airpore.cpp:573-580), on the East face from its rows (they
    // are complete when the node is not)
    auto sample = [&](const T *p, int step, bool rows) {
        for (int r = e; r < G.nrec; r += CN) {
            const long long q = b.rec_idx[r];
            if (q < 0) {
                if (c0 == 0) rec_out[(size_t)step * G.nrec + r] = 0.0;
                continue;
            }
            const int rk = (int)(q / P), rn = (int)(q - (long long)rk * P), rc = pnz + rk;
            if (rc < c0 || rc >= c1) continue;
            const int x = (rc - lo) * P + rn;
            T s = p[x];
            if (rows && rn >= P - nx) s = T(15.0 / 8.0) * p[x - nx] - T(5.0 / 4.0) * p[x - 2 * nx] + T(3.0 / 8.0) * p[x - 3 * nx];
            double v = (double)s;
            if (fabs(v) < 1.0e-100) v = 0.0;
            rec_out[(size_t)step * G.nrec + r] = v;
        }
    };
    const T dt = g.dt;
    const int nrec = G.nrec;
    __syncthreads();
    if (nrec) {
        sample(F[0][3], 0, false);
        __syncthreads();
    }
    for (int s = 0; s < nsteps; ++s) {
        T(&o)[4][CN] = F[s & 1];
        T(&w)[4][CN] = F[(s & 1) ^ 1];
        const Lay<T> l0{};
        // the planes that the owned ones still depend on
        const int reach = nsteps - s + 2;
        const bool used = live && c >= c0 - reach && c < c1 + reach;
        if (used && !east) {
            const T pc = o[3][es];
            T p;
            n.uc = o[0][es]; n.vc = o[1][es]; n.wc = o[2][es];
            n.u_ip = o[0][es + 1]; n.v_jp = o[1][es + nx]; n.w_kp = o[2][up];
            if (sground) {
                const T div = n.mX * g.dxi * (n.u_ip - n.uc) + n.mY * g.dyi * (n.v_jp - n.vc) + n.mZ * g.dzi * (n.w_kp - n.wc);
                p = pc + (-(T)b.g_gama * div);
            } else if (sair) {
                n.pc = pc;
                T ddx, ddy, dwz;
                T r = dp_core<T, 0, false, false>(a, n, ddx, ddy, dwz);
                if (lay) {
                    QP<T> x{}, y{}, z{};
                    z.u0 = Q[0][es]; z.ui = Q[0][es + 1];
                    z.v0 = Q[1][es]; z.vj = Q[1][es + nx];
                    r = row_dp_layers<T, false, false, false, true>(a, n, l0, l0, lz, x, y, z, pc, ddx, ddy, dwz, r);
                }
                p = pc + r;
            } else {
                const T div = ((n.mX * h.dxi) * (n.u_ip - n.uc) + (n.mY * h.dyi) * (n.v_jp - n.vc)) + (n.mZ * h.dzi) * (n.w_kp - n.wc);
                p = pc + (-A.pgama) * div;
            }
            w[3][e] = p;
            if (has) Q[3][e] += dt * p;
        }
        __syncthreads();
        if (used) {
            T f[3];
            const T uc = o[0][es], vc = o[1][es], wc = o[2][es];
            n.uc = uc; n.vc = vc; n.wc = wc;
            n.pc = w[3][es]; n.p_im = w[3][es - 1]; n.p_jm = w[3][es - nx]; n.p_km = w[3][dn];
            if (sground) {
                const T ib = (T)b.g_ib, eff = (T)b.g_eff;
                const T gx = n.mX * (n.pc - n.p_im) * g.dxi, gy = n.mY * (n.pc - n.p_jm) * g.dyi;
                f[0] = uc + (T(-1.0) * ib * b.dt * eff * gx + uc * ib - uc);
                f[1] = vc + (T(-1.0) * ib * b.dt * eff * gy + vc * ib - vc);
                const int np = jp * nx + ip;
                const double(&ho)[8][kColPlane] = psi[s & 1];
                double temp_psi = 0;
                for (int q = 0; q < b.gK; ++q) temp_psi += b.gdecay[q] * ho[q][np];
                const double hist = b.gZinf * temp_psi;
                const double wd = ((double)wc - b.gcpl * ((double)n.pc - hist)) * b.g_ib / (1.0 + b.g_ib * b.gcpl * b.gzi);
                f[2] = (T)wd;
                const double vg = -wd;
                if (inner)
                    for (int q = 0; q < b.gK; ++q)
                        psi[(s & 1) ^ 1][q][nd] = b.gdecay[q] * ho[q][np] + (b.ggain[q] * vg) * b.gtb;
            } else if (sair) {
                T gpx, gpy, gpz, du, dv, dw;
                duvw_core<T, 0, false, false>(a, n, gpx, gpy, gpz, du, dv, dw);
                if (lay) {
                    QV<T> x{}, y{}, z{};
                    z.p0 = Q[3][es]; z.pi = Q[3][es - 1]; z.pj = Q[3][es - nx];
                    row_duvw_layers<T, false, false, false, true>(a, n, l0, l0, lz, x, y, z, uc, vc, wc, gpx, gpy, gpz, du, dv, dw);
                }
                f[0] = uc + du; f[1] = vc + dv; f[2] = wc + dw;
            } else {
                const T gx = (n.mX * (n.pc - n.p_im)) * h.dxi, gy = (n.mY * (n.pc - n.p_jm)) * h.dyi, gz = (n.mZ * (n.pc - n.p_km)) * h.dzi;
                const T cf = ((T(-1.0) * A.pinvb) * h.dt) * A.peff;
                f[0] = uc + ((cf * gx + uc * A.pinvb) - uc);
                f[1] = vc + ((cf * gy + vc * A.pinvb) - vc);
                f[2] = wc + ((cf * gz + wc * A.pinvb) - wc);
            }
            if (xface) f[0] = T(0);
            if (west || east) f[1] = T(0);
            if (rigid) f[2] = T(0);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                w[q][e] = f[q];
                if (has) Q[q][e] += dt * f[q];
            }
            if (east) {
                const T pe = T(15.0 / 8.0) * w[3][e - nx] - T(5.0 / 4.0) * w[3][e - 2 * nx] + T(3.0 / 8.0) * w[3][e - 3 * nx];
                w[3][e] = pe;
                if (has) Q[3][e] += dt * pe;
            }
        }
        if (nrec && s + 1 < nsteps) sample(w[3], s + 1, true);
        __syncthreads();
    }
    if (!mine) return;
    const T(&r)[4][CN] = F[nsteps & 1];
    const Grid<T> &d = air ? g : h;
    d.unn[ge] = r[0][e]; d.vnn[ge] = r[1][e]; d.wnn[ge] = r[2][e]; d.pnn[ge] = r[3][e];
    if (has)
#pragma unroll
        for (int f = 0; f < 4; ++f) A.q[2].n[f][qe] = Q[f][e];
    if (G.ground && air && k == 0 && inner)
        for (int q = 0; q < b.gK; ++q) b.gpsi_new[(size_t)q * P + nd] = psi[nsteps & 1][q][nd];
}

}  // namespace

// Planes a workgroup owns, planes of halo and steps per launch.  Halo work costs nothing while
// the owned planes' workgroups still find a CU each, so as few planes are owned as a launch of
// 240 workgroups allows.
ColPlan col_plan(int nx, int ny, int nz, int pnz)
{
    ColPlan p{};
    if ((long long)nx * ny > kColPlane || nx < 3 || ny < 5 || nz < 3 || (pnz && pnz < 3)) return p;
    const int W = CN / (nx * ny), C = nz + pnz, own = (C + 239) / 240;
    const int steps = (W - own) / 2 - 3;
    if (steps < 2) return p;
    p.own = own; p.halo = steps + 3; p.steps = steps; p.blocks = (C + own - 1) / own;
    return p;
}
template <typename T> void launch_col(const RowArgs<T> *ad, const ColPlan &p, int nsteps, double *rec, hipStream_t s)
{
    hipLaunchKernelGGL((k_col<T>), dim3((unsigned)p.blocks), dim3(CN), 0, s, ad, p.own, p.halo, nsteps, rec);
}
template void launch_col<double>(const RowArgs<double> *, const ColPlan &, int, double *, hipStream_t);
template void launch_col<float>(const RowArgs<float> *, const ColPlan &, int, double *, hipStream_t);

}  // namespace lee
