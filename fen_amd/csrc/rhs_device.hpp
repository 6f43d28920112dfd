// rhs_device.hpp -- the Poisson right-hand side at one cell, as the x
// transforms load it (div_r2c_kernel, plane_fwd_kernel): first the loads of a
// whole row, then its arithmetic, with a scheduling barrier between.  Left to
// the compiler the loads stood among the divisions, and a thread waited for
// memory several times per row (128^2: 6.0 -> 5.5 us, 256^3: 118 -> 112).
#pragma once

#include "fen_internal.hpp"

namespace fen {

// MODE 0: div(u*) rho / dt of the ghosted velocity; 1: `u` itself (strides sx,
// sy, ghost level gl); 2 (FP64): p + scale div(u, v, w) of interior arrays,
// periodic in every direction (the discrete adjoint's).  (i, j, k) from 1.
template <class R, int MODE, int D3, class A>
__device__ __forceinline__ void rhs_load(const A &a, R (&f)[7], int i, int j, int k)
{
    if constexpr (MODE == 2) {
        const long nx = a.b.nx, ny = a.b.ny;
        const long row = nx * ((j - 1) + ny * (k - 1));
        const long rowj = nx * ((j == 1 ? ny - 1 : j - 2) + ny * (k - 1));
        const long rowk = nx * ((j - 1) + ny * (k == 1 ? a.b.nz - 1 : k - 2));
        const int x = i - 1, xm = i == 1 ? (int)nx - 1 : i - 2;
        f[0] = a.u[row + x];
        f[1] = a.u[row + xm];
        f[2] = a.v[row + x];
        f[3] = a.v[rowj + x];
        f[4] = a.w[row + x];
        f[5] = a.w[rowk + x];
        f[6] = a.p[row + x];
    } else if constexpr (MODE == 1) {
        f[0] = a.u[(i - 1 + a.gl) + a.sx * (j - 1 + a.gl) + a.sy * (k - 1 + a.gl)];
    } else {
        const long g = a.b.g(i, j, k);
        f[0] = a.u[g];
        f[1] = a.u[g - 1];
        f[2] = a.v[g];
        f[3] = a.v[g - a.b.gx];
        if constexpr (D3) {
            f[4] = a.w[g];
            f[5] = a.w[g - a.b.gxy];
        }
    }
}

template <class R, int MODE, int D3, class A> __device__ __forceinline__ double rhs_value(const A &a, const R (&f)[7])
{
    if constexpr (MODE == 1) return (double)f[0];
    double d = ((double)f[0] - (double)f[1]) * a.id + ((double)f[2] - (double)f[3]) * a.id;
    if constexpr (D3) d = d + ((double)f[4] - (double)f[5]) * a.id;
    if constexpr (MODE == 2) return (double)f[6] + a.scale * d;
    else return d * a.rho / a.dt;
}

}  // namespace fen
