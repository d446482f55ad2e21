// lee_core.h -- per-point arithmetic shared by the stencil kernels: the inverse metric and the
// interior increments of the air fields.  Every kernel that advances a point calls these, so
// all launch shapes compute the same bits.
#pragma once

#include <type_traits>

#include "lee_kernels.h"

namespace lee {

namespace {

template <typename T> __device__ __forceinline__ void metric(const Grid<T> &g, int i, int j, int k, T &mX, T &mY, T &mZ)
{
    if constexpr (std::is_same<T, double>::value) {
        // Jacobian of calculation_2D.cpp:424-430 and Geo_over_var (df_over_var.cpp:5-9)
        double xx = g.mx[i], yy = g.my[j], zz = g.mz[k];
        double J = 1.0 / (xx * yy * zz);
        mX = (yy * zz) * J;
        mY = (xx * zz) * J;
        mZ = (xx * yy) * J;
    } else {
        mX = g.mx[i]; mY = g.my[j]; mZ = g.mz[k];
    }
}

// Terrain-following grid: X_over_x, Y_over_y as in the reference, Z_over_z = Zz[k]*sh(i,j),
// Z_over_x = hx(i,j)*tk[k], Z_over_y = hy(i,j)*tk[k].  Of the nine inverse-metric terms of
// Geo_over_var (df_over_var.cpp:5-9) five are non-zero: xX, yY, zZ and the cross terms
// zX = -(Yy*Zx)*J, zY = -(Xx*Zy)*J.  The tables hold X_over_x ... (not reciprocals) in both
// precisions.
template <typename T> __device__ __forceinline__ void metric_terrain(const Grid<T> &g, int i, int j, int k, T &mX, T &mY,
                                                                     T &mZ, T &zX, T &zY)
{
    const size_t c = (size_t)i + (size_t)g.nx * j;
    const T xx = g.mx[i], yy = g.my[j], zz = g.mz[k] * g.tsh[c];
    const T Zx = g.thx[c] * g.ttk[k], Zy = g.thy[c] * g.ttk[k];
    const T J = T(1) / (xx * yy * zz);
    mX = (yy * zz) * J;
    mY = (xx * zz) * J;
    mZ = (xx * yy) * J;
    zX = (-(yy * Zx)) * J;
    zY = (-(xx * Zy)) * J;
}

// ------------------------------------------------------------------------------------
// The interior arithmetic of the pressure and velocity increments for the mean flows of
// velocity_method 0 and 7 (none, or V along y only), from the point's neighbour values.  The
// one-point stencils below and the four-point form of the RK4 stage both call these, so every
// launch shape computes the same bits.
// ------------------------------------------------------------------------------------
template <typename T> struct Nb {
    T mX, mY, mZ, zX, zY;                        // inverse metric (zX = zY = 0 on a flat grid)
    T pc, p_im, p_jp, p_jm, p_kp, p_km;          // p and its neighbours (i-1, j+-1, k+-1)
    T uc, u_ip, u_jp, u_jm, u_kp, u_km;          // u
    T vc, v_jp, v_jm, v_kp, v_km;                // v
    T wc, w_jp, w_jm, w_kp, w_km;                // w
    T Vc, V_ip, V_im, V_jp, V_jm, V_kp, V_km;    // mean flow along y
};

// dt*R_p without the layer terms (air.cpp:1953-2043); also the damped terms ddx, ddy and
// the difference dwz the layer terms use.
template <typename T, int WM, bool TERRAIN, bool CEN>
__device__ __forceinline__ T dp_core(const AirArgs<T> &a, const Nb<T> &n, T &ddx, T &ddy, T &dwz)
{
    const Grid<T> &g = a.g;
    const T dxi = g.dxi, dyi = g.dyi, dzi = g.dzi, dt = g.dt;
    const T mX = n.mX, mY = n.mY, mZ = n.mZ, zX = n.zX, zY = n.zY, pc = n.pc;
    const T dux = n.u_ip - n.uc;
    const T dvy = n.v_jp - n.vc;
    dwz = n.w_kp - n.wc;
    T duz = T(0), dvz = T(0);
    T div;
    if constexpr (TERRAIN) {
        duz = n.u_kp - n.uc;
        dvz = n.v_kp - n.vc;
        div = (((((mX * dux) * dxi) + ((zX * duz) * dzi)) + ((mY * dvy) * dyi)) + ((zY * dvz) * dzi)) + ((mZ * dwz) * dzi);
    } else {
        div = (((mX * dux) * dxi) + ((mY * dvy) * dyi)) + ((mZ * dwz) * dzi);
    }
    ddx = (mX * dux) * dxi;
    ddy = (mY * dvy) * dyi;
    if constexpr (TERRAIN) {
        ddx = ddx + (zX * duz) * dzi;
        ddy = ddy + (zY * dvz) * dzi;
    }
    T r;
    if constexpr (WM == 2) {
        // mean flow along y only (U = W = 0): the terms with U or W are exact zeros
        const T Vc = n.Vc;
        const T c2 = ((Vc * mY) * dyi) * dt;
        T VY = ((mY * (n.V_jp - n.V_jm)) * dyi) * T(0.5);
        if constexpr (CEN) r = -(c2 * ((n.p_jp - n.p_jm) * T(0.5)));
        else r = -(c2 * (pc - n.p_jm));
        if constexpr (TERRAIN) {
            const T c3 = ((Vc * zY) * dzi) * dt;
            VY = VY + ((zY * (n.V_kp - n.V_km)) * dzi) * T(0.5);
            if constexpr (CEN) r = r - c3 * ((n.p_kp - n.p_km) * T(0.5));
            else r = r - c3 * (pc - n.p_km);
        }
        r += (((-a.gam) * pc) * dt) * VY;
        r += (((-a.gam) * a.Pav) * dt) * div;
    } else {
        r = (((-a.gam) * a.Pav) * dt) * div;
    }
    return r;
}

// dt*R_u, dt*R_v, dt*R_w without the layer terms (air.cpp:1476-1578); also the pressure
// gradients gpx, gpy, gpz the layer terms use.
template <typename T, int WM, bool TERRAIN, bool CEN>
__device__ __forceinline__ void duvw_core(const AirArgs<T> &a, const Nb<T> &n, T &gpx, T &gpy, T &gpz, T &du, T &dv,
                                          T &dw)
{
    const Grid<T> &g = a.g;
    const T dxi = g.dxi, dyi = g.dyi, dzi = g.dzi, dt = g.dt, Aav = a.Aav;
    const T mX = n.mX, mY = n.mY, mZ = n.mZ, zX = n.zX, zY = n.zY, pc = n.pc;
    const T bpz = pc - n.p_km;
    gpx = (mX * (pc - n.p_im)) * dxi;
    gpy = (mY * (pc - n.p_jm)) * dyi;
    gpz = (mZ * bpz) * dzi;
    if constexpr (TERRAIN) {
        gpx = gpx + (zX * bpz) * dzi;
        gpy = gpy + (zY * bpz) * dzi;
    }
    const T uc = n.uc, vc = n.vc, wc = n.wc;
    if constexpr (WM == 2) {
        // mean flow along y only (U = W = 0): the terms with U or W or their gradients vanish
        const T Vc = n.Vc;
        const T c2 = ((Vc * mY) * dyi) * dt;
        T VX = ((mX * (n.V_ip - n.V_im)) * dxi) * T(0.5);
        T VY = ((mY * (n.V_jp - n.V_jm)) * dyi) * T(0.5);
        const T VZ = ((mZ * (n.V_kp - n.V_km)) * dzi) * T(0.5);
        // d/dY (and d/dZ over terrain) of one component: forward (reference) or central
        auto d1 = [&](T fp, T fm, T fc) {
            if constexpr (CEN) return (fp - fm) * T(0.5);
            else return fp - fc;
        };
        du = -(c2 * d1(n.u_jp, n.u_jm, uc));
        dv = -(c2 * d1(n.v_jp, n.v_jm, vc));
        dw = -(c2 * d1(n.w_jp, n.w_jm, wc));
        if constexpr (TERRAIN) {
            const T c3 = ((Vc * zY) * dzi) * dt;
            VX = VX + ((zX * (n.V_kp - n.V_km)) * dzi) * T(0.5);
            VY = VY + ((zY * (n.V_kp - n.V_km)) * dzi) * T(0.5);
            du = du - c3 * d1(n.u_kp, n.u_km, uc);
            dv = dv - c3 * d1(n.v_kp, n.v_km, vc);
            dw = dw - c3 * d1(n.w_kp, n.w_km, wc);
        }
        du += ((-Aav) * dt) * gpx;
        dv += (((-uc) * VX) * dt - (vc * VY) * dt) - (wc * VZ) * dt;
        dv += ((-Aav) * dt) * gpy;
        dw += ((-Aav) * dt) * gpz;
    } else {
        du = ((-Aav) * dt) * gpx;
        dv = ((-Aav) * dt) * gpy;
        dw = ((-Aav) * dt) * gpz;
    }
}

}  // namespace

}  // namespace lee
