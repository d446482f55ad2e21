// lee_faces.h -- per-node arithmetic of the face conditions shared by the face passes
// (lee_bc.hip) and the row kernels (lee_fb.hip): the ground interface plane and the East TDBC.
#pragma once

#include "lee_kernels.h"

namespace lee {

namespace {

template <typename T> __device__ __forceinline__ size_t gidx(const Grid<T> &g, int i, int j, int k)
{
    return (size_t)i + (size_t)g.nx * ((size_t)j + (size_t)g.ny * k);
}

// Ground impedance (extension): the plane k = 0 is the ground's interface plane, as the
// porous ground's top plane is when the air reads it through the interface copy
// (calculation_2D.cpp:878-886).  Its interior nodes are stencil output of the porous
// equations of the ground's top material (porous.cpp:77-143 with porous.cpp:44-50) -- the
// faces N E W F B then treat its edge nodes as on every other plane, and there is no South
// face.  The normal velocity (half a cell below the plane) follows the porous momentum
// equation with the pressure half a cell further down given by the impedance through the
// TDBC recursion of calculation_2D.cpp:986-1028 with K poles.  The plane's metric is the
// porous top plane's: gmx[i] = 1/X_over_x, gmy[j] = 1/Y_over_y, gmz = 1/Z_over_z of the plane
// k = 1, and on the terrain-following grid the cross terms zX, zY of the inverse Jacobian per
// node (the tables of gter) of a layer shifted rigidly with the ground, as porous.cpp's grid is
// under airpore.cpp's hills, not the air column's compressed metric.  The plane's z derivatives
// are one-sided towards k = 1.  With no hill every term reduces to the flat closure's bit for
// bit (the cross terms are zeros).
template <typename T> __device__ __forceinline__ T ground_p(const BCArgs<T> &a, int i, int j)
{
    const Grid<T> &g = a.air;
    const size_t e = gidx(g, i, j, 0);
    const T ex = (T)a.gmx[i], ey = (T)a.gmy[j], ez = (T)a.gmz;
    T div;
    if (a.gter) {
        const size_t c = (size_t)i + (size_t)g.nx * j, n2 = (size_t)g.nx * g.ny;
        const T zX = (T)a.gter[c], zY = (T)a.gter[n2 + c];
        const T dux = g.un[gidx(g, i + 1, j, 0)] - g.un[e], duz = g.un[gidx(g, i, j, 1)] - g.un[e];
        const T dvy = g.vn[gidx(g, i, j + 1, 0)] - g.vn[e], dvz = g.vn[gidx(g, i, j, 1)] - g.vn[e];
        div = ((ex * g.dxi * dux + zX * g.dzi * duz) + (ey * g.dyi * dvy + zY * g.dzi * dvz)) +
              ez * g.dzi * (g.wn[gidx(g, i, j, 1)] - g.wn[e]);
    } else {
        div = ex * g.dxi * (g.un[gidx(g, i + 1, j, 0)] - g.un[e]) + ey * g.dyi * (g.vn[gidx(g, i, j + 1, 0)] - g.vn[e]) +
              ez * g.dzi * (g.wn[gidx(g, i, j, 1)] - g.wn[e]);
    }
    return g.pn[e] + (-(T)a.g_gama * div);
}

// East TDBC velocity from the final boundary pressure and the history of the previous step
// (calculation_2D.cpp:1019-1028).
template <typename T> __device__ __forceinline__ double tdbc_v(const BCArgs<T> &a, int i, int k)
{
    const Grid<T> &g = a.air;
    const double *P = a.psi_old + ((size_t)i + (size_t)g.nx * k) * 6;
    double temp_psi = 0;
#pragma unroll
    for (int q = 0; q < 6; ++q) temp_psi += a.decay[q] * P[q];
    return a.inv * ((double)g.pnn[gidx(g, i, g.ny - 1, k)] / a.Zinf - temp_psi);
}

// Ground plane velocities of interior node (i, j) from the final pressures of the plane:
// tangential components by the porous momentum equation, the normal one (double: it feeds
// the FP64 histories) with the impedance's pressure half a cell below it,
//   w' = ib (w - cpl (p' - p_h)),  p_h = Zinf (1 + tb sum a) v + Zinf sum_k e^{-r_k tb} Psi_k,
// v = -w', solved for w'.
template <typename T> __device__ __forceinline__ double ground_w_of(const BCArgs<T> &a, int i, int j, double temp_psi)
{
    const Grid<T> &g = a.air;
    const size_t e = gidx(g, i, j, 0);
    const double hist = a.gZinf * temp_psi;
    return ((double)g.wn[e] - a.gcpl * ((double)g.pnn[e] - hist)) * a.g_ib / (1.0 + a.g_ib * a.gcpl * a.gzi);
}

// The ground histories are pole-major, Psi_q of node (i, j) at q * nx * ny + i + nx * j, so
// that each pole's reads and writes of a wave are contiguous.
template <typename T> __device__ __forceinline__ double ground_w(const BCArgs<T> &a, int i, int j)
{
    const size_t node = (size_t)i + (size_t)a.air.nx * j, nn = (size_t)a.air.nx * a.air.ny;
    double temp_psi = 0;
    for (int q = 0; q < a.gK; ++q) temp_psi += a.gdecay[q] * a.gpsi_old[q * nn + node];
    return ground_w_of(a, i, j, temp_psi);
}

template <typename T> __device__ __forceinline__ T ground_vel(const BCArgs<T> &a, int c, int i, int j)
{
    const Grid<T> &g = a.air;
    const size_t e = gidx(g, i, j, 0);
    const T ib = (T)a.g_ib, dt = a.dt, eff = (T)a.g_eff;
    // terrain: d/dX = ex d/dx + zX d/dz, d/dY = ey d/dy + zY d/dz with d/dz one-sided to
    // k = 1; on a flat grid the cross term is absent
    T pz = T(0), zX = T(0), zY = T(0);
    if (a.gter) {
        const size_t q = (size_t)i + (size_t)g.nx * j, n2 = (size_t)g.nx * g.ny;
        pz = (g.pnn[gidx(g, i, j, 1)] - g.pnn[e]) * g.dzi;
        zX = (T)a.gter[q];
        zY = (T)a.gter[n2 + q];
    }
    if (c == 0) {
        const T ex = (T)a.gmx[i];
        T gx = ex * (g.pnn[e] - g.pnn[gidx(g, i - 1, j, 0)]) * g.dxi;
        if (a.gter) gx = gx + zX * pz;
        return g.un[e] + (T(-1.0) * ib * dt * eff * gx + g.un[e] * ib - g.un[e]);
    }
    if (c == 1) {
        const T ey = (T)a.gmy[j];
        T gy = ey * (g.pnn[e] - g.pnn[gidx(g, i, j - 1, 0)]) * g.dyi;
        if (a.gter) gy = gy + zY * pz;
        return g.vn[e] + (T(-1.0) * ib * dt * eff * gy + g.vn[e] * ib - g.vn[e]);
    }
    return (T)ground_w(a, i, j);
}

}  // namespace

}  // namespace lee
