// mf_kernels.hip -- the two-phase step of FEN's MF build on the GPU, 2-D,
// FP64: MTHINC volume of fluid (Ii et al. 2012; reference
// src/volume_of_fluid.f90), material properties (src/multiphase.f90:126-140),
// and the momentum right-hand side with variable density and viscosity, CSF
// surface tension and the Dodd & Ferrante pressure splitting
// (src/navier_stokes.f90:140-213, 384-501).  One thread per cell; the
// expressions keep the reference's evaluation order (the library is built
// with -ffp-contract=off).
#include <stdexcept>

#include "fen_internal.hpp"

namespace fen {

namespace {

constexpr int kBX = 16, kBY = 16;
constexpr double kSmall = 1.0e-14;   // global_mod small (src/global.f90:16)
constexpr double kCut = 1.0e-8;      // cut (src/volume_of_fluid.f90:37)

__device__ __forceinline__ double gauss_rp() { return 0.5 * (1.0 + 1.0 / sqrt(3.0)); }
__device__ __forceinline__ double gauss_rm() { return 0.5 * (1.0 - 1.0 / sqrt(3.0)); }

struct Surf {
    double cx, cy, a10, a01, a20, a02;
};

// P(x, y), Eq. 9 of Ii et al. (src/volume_of_fluid.f90:387-398)
__device__ __forceinline__ double surf_p(const Surf &q, double x, double y)
{
    return ((q.cx * q.a20 * (x * x) + q.cy * q.a02 * (y * y)) + q.a10 * x) + q.a01 * y;
}

__device__ __forceinline__ Surf cell_surface(double nx, double ny, double lx, double ly)
{
    Surf q;
    if (fabs(nx) == fmax(fabs(nx), fabs(ny))) { q.cx = 0.0; q.cy = 1.0; }
    else { q.cx = 1.0; q.cy = 0.0; }
    q.a10 = nx - 0.5 * q.cx * lx;
    q.a01 = ny - 0.5 * q.cy * ly;
    q.a20 = 0.5 * q.cx * lx;
    q.a02 = 0.5 * q.cy * ly;
    return q;
}

// The MF fields' ghosts are copies (periodic images, or the neighbour at a
// Neumann wall; src/volume_of_fluid.f90:54-219, src/multiphase.f90:44-120), by
// each face's own rule: an axis may have one periodic face and one wall.
struct MFCopies {
    int face[4];   // COPY_PERIODIC or COPY_MIRROR: left, right, bottom, top
};

// Stores n fields' values of cell (i, j) and the ghosts that copy them.
template <int NF>
__device__ __forceinline__ void put_copies(const Box &b, const MFCopies &m, int i, int j, double *const (&f)[NF],
                                           const double (&v)[NF])
{
    int id[3], jd[3];
    const int ni = copy_rows(i, b.nx, m.face[0], m.face[1], id), nj = copy_rows(j, b.ny, m.face[2], m.face[3], jd);
    for (int y = 0; y < nj; y++)
        for (int x = 0; x < ni; x++) {
            const long g = b.g(id[x], jd[y], 1);
#pragma unroll
            for (int q = 0; q < NF; q++) f[q][g] = v[q];
        }
}

struct VofArgs {
    MFCopies copies;
    Box b;
    double delta, id, id2, beta, dt;
    const double *vof;
    double *dd, *curv, *nrx, *nry, *lx, *ly;
};

// compute_norm (src/volume_of_fluid.f90:299-383) and the cell loop of
// get_h_from_vof (:223-295) in one pass: the normalisation needs only the
// cell's own normal and curvature terms.  (h itself, the smoothed indicator, is
// formed by the reference and read by nothing on this path.)
__global__ __launch_bounds__(kBX *kBY) void vof_reconstruct_kernel(VofArgs a)
{
    const int i = blockIdx.x * kBX + threadIdx.x % kBX + 1, j = blockIdx.y * kBY + threadIdx.x / kBX + 1;
    if (i > a.b.nx || j > a.b.ny) return;
    const long g = a.b.g(i, j, 1), sj = a.b.gx;
    const double *F = a.vof + g;
    auto V = [&](int di, int dj) { return F[di + dj * sj]; };
    const double id = a.id;
    double mx[4], my[4];
    mx[0] = 0.5 * (V(0, -1) + V(0, 0) - V(-1, -1) - V(-1, 0)) * id;
    mx[1] = 0.5 * (V(0, 0) + V(0, 1) - V(-1, 0) - V(-1, 1)) * id;
    mx[2] = 0.5 * (V(1, 0) + V(1, 1) - V(0, 0) - V(0, 1)) * id;
    mx[3] = 0.5 * (V(1, -1) + V(1, 0) - V(0, -1) - V(0, 0)) * id;
    const double mxc = 0.25 * (mx[0] + mx[1] + mx[2] + mx[3]);
    my[0] = 0.5 * (V(-1, 0) + V(0, 0) - V(-1, -1) - V(0, -1)) * id;
    my[1] = 0.5 * (V(-1, 1) + V(0, 1) - V(-1, 0) - V(0, 0)) * id;
    my[2] = 0.5 * (V(0, 1) + V(1, 1) - V(0, 0) - V(1, 0)) * id;
    my[3] = 0.5 * (V(0, 0) + V(1, 0) - V(0, -1) - V(1, -1)) * id;
    const double myc = 0.25 * (my[0] + my[1] + my[2] + my[3]);
    double nxs[4], nys[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        nxs[q] = mx[q] / sqrt(mx[q] * mx[q] + my[q] * my[q] + kSmall);
        nys[q] = my[q] / sqrt(mx[q] * mx[q] + my[q] * my[q] + kSmall);
    }
    const double nx = mxc / sqrt(mxc * mxc + myc * myc + kSmall);
    const double ny = myc / sqrt(mxc * mxc + myc * myc + kSmall);
    const double lx = 0.5 * a.delta * (nxs[3] + nxs[2] - nxs[1] - nxs[0]);   // quadratic reconstruction
    const double ly = 0.5 * a.delta * (nys[1] + nys[2] - nys[0] - nys[3]);
    const double f = V(0, 0);
    double *const out[6] = {a.nrx, a.nry, a.lx, a.ly, a.curv, a.dd};
    double val[6] = {nx, ny, lx, ly, -(lx + ly) * a.id2, 0.0};
    if (f <= kCut || f >= (1.0 - kCut)) {
        put_copies(a.b, a.copies, i, j, out, val);
        return;
    }
    const Surf q = cell_surface(nx, ny, lx, ly);
    const double beta = a.beta, rp = gauss_rp(), rm = gauss_rm();
    const double A = (1.0 - q.cx) * exp(2.0 * beta * q.a10) + (1.0 - q.cy) * exp(2.0 * beta * q.a01);
    const double Bp = (1.0 - q.cx) * exp(2.0 * beta * surf_p(q, 0.0, rp)) +
                      (1.0 - q.cy) * exp(2.0 * beta * surf_p(q, rp, 0.0));
    const double Bm = (1.0 - q.cx) * exp(2.0 * beta * surf_p(q, 0.0, rm)) +
                      (1.0 - q.cy) * exp(2.0 * beta * surf_p(q, rm, 0.0));
    const double Q = (1.0 - q.cx) * exp(2.0 * beta * q.a10 * (2.0 * f - 1.0)) +
                     (1.0 - q.cy) * exp(2.0 * beta * q.a01 * (2.0 * f - 1.0));
    const double aa = A * Bm * Bp * (A - Q);
    const double bb = A * (Bp + Bm) * (1.0 - Q);
    const double cc = 1.0 - A * Q;
    const double x1 = (-bb + sqrt(bb * bb - 4.0 * aa * cc)) / (2.0 * aa);   // solve_quadratic (:402-416)
    const double x2 = (-bb - sqrt(bb * bb - 4.0 * aa * cc)) / (2.0 * aa);
    val[5] = log(fmax(x1, x2)) / (2.0 * beta);
    put_copies(a.b, a.copies, i, j, out, val);
}

struct SweepArgs {
    MFCopies copies;
    Box b;
    double delta, beta, dt;
    const double *vof, *dd, *nrx, *nry, *lx, *ly;   // the current reconstruction; vof is swept
    const double *u, *v;
    double *out;                                    // first sweep: vof after it; second: the new vof
    // the second sweep's, if `rho` is set: material properties and p_hat of the new vof
    double rho0, rho1, mu0, mu1, dt_hat, dt_o;
    const double *p, *p_o;
    double *rho, *mu, *p_hat;
};

// compute_flux (src/volume_of_fluid.f90:548-632): flux through the high face
// of cell (i, j) along DIR with face velocity u.
template <int DIR> __device__ double face_flux(const SweepArgs &a, int i, int j, double u)
{
    const double delta = a.delta, dt = a.dt, beta = a.beta;
    double xa, xb, ya, yb;
    int sgn, ii = i, jj = j;
    if (DIR == 1) {
        if (u >= 0.0) { xa = 1.0 - dt * u / delta; xb = 1.0; sgn = 1; }
        else { xa = 0.0; xb = -dt * u / delta; sgn = -1; ii = i + 1; }
        ya = 0.0; yb = 1.0;
    } else {
        xa = 0.0; xb = 1.0;
        if (u >= 0.0) { ya = 1.0 - dt * u / delta; yb = 1.0; sgn = 1; }
        else { ya = 0.0; yb = -dt * u / delta; sgn = -1; jj = j + 1; }
    }
    const long g = a.b.g(ii, jj, 1);
    const double f = a.vof[g];
    if (f <= kCut || f >= (1.0 - kCut)) return (double)sgn * delta * f * (xb - xa) * (yb - ya);
    const Surf q = cell_surface(a.nrx[g], a.nry[g], a.lx[g], a.ly[g]);
    const double d0 = a.dd[g];
    // Num_Int of An_Int at the two Gauss points (src/volume_of_fluid.f90:636-661):
    // analytic along x (cx = 0) or along y, two points along the other.  One
    // loop for both directions and points: inlined eight times over, the cosh
    // made 30 KB of code, fetched cold by every launch.
    const bool along_x = q.cx == 0.0;
    const double lo = along_x ? xa : ya, hi = along_x ? xb : yb;         // analytic direction
    const double ql = along_x ? ya : xa, qh = along_x ? yb : xb;         // the other
    const double cf = along_x ? q.a10 : q.a01;
    double sum = 0.0;
#pragma unroll 1
    for (int n = 0; n < 2; n++) {
        const double t = (n == 0 ? gauss_rm() : gauss_rp()) * (ql + qh);
        double c[2];
#pragma unroll 1
        for (int m = 0; m < 2; m++) {
            const double x = m == 0 ? hi : lo;
            c[m] = cosh(beta * (surf_p(q, along_x ? x : t, along_x ? t : x) + d0));
        }
        sum = sum + 0.5 * (hi - lo + 1.0 / (cf * beta) * log(c[0] / c[1]));
    }
    return (double)sgn * delta * (0.5 * sum * (qh - ql));
}

// rho and mu of a cell (src/multiphase.f90:133-134), and p_hat: 2 p - p_o at
// fixed dt (src/navier_stokes.f90:91), p_o + (dt + dt_o)(p - p_o)/dt_o with
// constant CFL (:89; `dt` > 0).
__device__ __forceinline__ double mix(double f, double a0, double a1) { return a1 * f + a0 * (1.0 - f); }
__device__ __forceinline__ double p_hat_of(double p, double p_o, double dt, double dt_o)
{
    return dt > 0.0 ? p_o + (dt + dt_o) * (p - p_o) / dt_o : 2.0 * p - p_o;
}

// One directional sweep of advect_vof (src/volume_of_fluid.f90:437-461).  The
// second one also finishes the advection, vof^{n+1} = vof2 - dt (vof_x du +
// vof_y dv) with the sweep order's weights (:463-470, :509-516; `vof` is vof1
// there), and forms rho, mu and p_hat of the new vof.  Every output leaves with
// its ghosts.  (The finish, the properties, a copy of vof1 and six ghost fills
// were launches of 4 us each, as long as the sweep of a 128 x 512 grid's cells
// themselves.)
//
// One thread per face of the workgroup's 16 x 16 cells along DIR (17 rows of
// faces), each formed once and read by the cell beyond it from LDS: a face of a
// mixed cell is some 800 dependent instructions (eight cosh, four log), and a
// thread that formed both of its cell's, all inlined, took 11 us a sweep, now 7.4
// (9 with the finish and the properties).
constexpr int kFaces = (kBX + 1) * kBY;
template <int DIR, int SECOND> __global__ __launch_bounds__(kFaces) void vof_sweep_kernel(SweepArgs a)
{
    static_assert(kBX == kBY, "square workgroups");
    __shared__ double flux[kFaces];
    // face row r (0: the low faces of the first cells) of line l; r is the slow index
    const int l = threadIdx.x % kBX, r = threadIdx.x / kBX;
    const int i0 = blockIdx.x * kBX, j0 = blockIdx.y * kBY;
    const int i = i0 + (DIR == 1 ? r : l + 1), j = j0 + (DIR == 1 ? l + 1 : r);   // the cell whose high face it is
    const double *vel = DIR == 1 ? a.u : a.v;
    if (i <= a.b.nx && j <= a.b.ny) flux[threadIdx.x] = face_flux<DIR>(a, i, j, vel[a.b.g(i, j, 1)]);
    __syncthreads();
    if (r == 0 || i > a.b.nx || j > a.b.ny) return;
    const long g = a.b.g(i, j, 1), sh = DIR == 1 ? 1 : a.b.gx;
    const double fp = flux[threadIdx.x], fm = flux[threadIdx.x - kBX];
    const double vof1 = a.vof[g];
    const double swept = (vof1 - (fp - fm) / a.delta) / (1.0 - a.dt * (vel[g] - vel[g - sh]) / a.delta);
    if constexpr (!SECOND) {
        double *const out[1] = {a.out};
        const double val[1] = {swept};
        put_copies(a.b, a.copies, i, j, out, val);
    } else {
        const double du = a.u[g] - a.u[g - 1], dv = a.v[g] - a.v[g - a.b.gx];
        // the direction swept first weighs with vof1
        const double vx = DIR == 2 ? vof1 : swept, vy = DIR == 2 ? swept : vof1;
        const double f = swept - a.dt * (vx * du / a.delta + vy * dv / a.delta);
        if (a.rho) {
            double *const out[4] = {a.out, a.rho, a.mu, a.p_hat};
            const double val[4] = {f, mix(f, a.rho0, a.rho1), mix(f, a.mu0, a.mu1),
                                   p_hat_of(a.p[g], a.p_o[g], a.dt_hat, a.dt_o)};
            put_copies(a.b, a.copies, i, j, out, val);
        } else {
            double *const out[1] = {a.out};
            const double val[1] = {f};
            put_copies(a.b, a.copies, i, j, out, val);
        }
    }
}

// rho and mu of the resident vof, with ghosts.
__global__ __launch_bounds__(kBX *kBY) void mf_fields_kernel(Box b, MFCopies copies, const double *vof, double rho0,
                                                             double rho1, double mu0, double mu1, double *rho,
                                                             double *mu)
{
    const int i = blockIdx.x * kBX + threadIdx.x % kBX + 1, j = blockIdx.y * kBY + threadIdx.x / kBX + 1;
    if (i > b.nx || j > b.ny) return;
    const double f = vof[b.g(i, j, 1)];
    double *const out[2] = {rho, mu};
    const double val[2] = {mix(f, rho0, rho1), mix(f, mu0, mu1)};
    put_copies(b, copies, i, j, out, val);
}

struct MFMomArgs {
    GhostDesc<double> gu, gv;   // u* and v*, left with their ghosts filled
    Box b;
    double id, dt, A, B, g0, g1, sigma, irhomin;
    const double *u, *v, *p, *p_hat, *rho, *mu, *vof, *curv, *s0, *s1;
    double *us, *vs, *dvo0, *dvo1;
};

// predicted_velocity_field with MF (src/navier_stokes.f90:140-213): advection
// (:261-353), variable-viscosity diffusion (:405-452), surface tension
// (:458-501), body force (:245-255), -grad p/rhof + A dv + B dv_o + g, the
// Dodd & Ferrante correction (:178-184), v* = v + dt RHS, dv_o = dv.
template <int SRC> __global__ __launch_bounds__(kBX *kBY) void mf_momentum_kernel(MFMomArgs a)
{
    const int i = blockIdx.x * kBX + threadIdx.x % kBX + 1, j = blockIdx.y * kBY + threadIdx.x / kBX + 1;
    if (i > a.b.nx || j > a.b.ny) return;
    const long g = a.b.g(i, j, 1), q = a.b.q(i, j, 1), sj = a.b.gx;
    const double id = a.id;
    auto U = [&](int di, int dj) { return a.u[g + di + dj * sj]; };
    auto V = [&](int di, int dj) { return a.v[g + di + dj * sj]; };
    auto M = [&](int di, int dj) { return a.mu[g + di + dj * sj]; };
    const double rfx = 0.5 * (a.rho[g + 1] + a.rho[g]);   // center_to_face (src/fields.f90:210-235)
    const double rfy = 0.5 * (a.rho[g + sj] + a.rho[g]);
    const double u0 = U(0, 0), v0 = V(0, 0);

    // advection, R = 0 - ...
    double rx, ry;
    {
        const double up = U(1, 0), um = U(-1, 0);
        const double uuip = 0.25 * ((up + u0) * (up + u0));
        const double uuim = 0.25 * ((um + u0) * (um + u0));
        const double uvjp = ((U(0, 1) + u0) * (V(1, 0) + v0)) * 0.25;
        const double uvjm = ((u0 + U(0, -1)) * (V(1, -1) + V(0, -1))) * 0.25;
        rx = (0.0 - (uuip - uuim) * id) - (uvjp - uvjm) * id;
        const double vuip = ((V(1, 0) + v0) * (U(0, 1) + u0)) * 0.25;
        const double vuim = ((v0 + V(-1, 0)) * (U(-1, 1) + U(-1, 0))) * 0.25;
        const double vp = V(0, 1), vm = V(0, -1);
        const double vvjp = 0.25 * ((vp + v0) * (vp + v0));
        const double vvjm = 0.25 * ((vm + v0) * (vm + v0));
        ry = (0.0 - (vuip - vuim) * id) - (vvjp - vvjm) * id;
    }
    // diffusion, div(2 mu D) with mu at cell centres
    {
        const double txxp = 2.0 * M(1, 0) * (U(1, 0) - U(0, 0)) * id;
        const double txxm = 2.0 * M(0, 0) * (U(0, 0) - U(-1, 0)) * id;
        const double dtxx = (txxp - txxm) * id;
        const double txyp = 0.25 * (M(0, 0) + M(1, 0) + M(0, 1) + M(1, 1)) *
                            ((U(0, 1) - U(0, 0)) * id + (V(1, 0) - V(0, 0)) * id);
        const double txym = 0.25 * (M(0, -1) + M(1, -1) + M(0, 0) + M(1, 0)) *
                            ((U(0, 0) - U(0, -1)) * id + (V(1, -1) - V(0, -1)) * id);
        const double dtxy = (txyp - txym) * id;
        rx = rx + (dtxx + dtxy) / rfx;
        const double tyxp = txyp;
        const double tyxm = 0.25 * (M(-1, 0) + M(0, 0) + M(-1, 1) + M(0, 1)) *
                            ((U(-1, 1) - U(-1, 0)) * id + (V(0, 0) - V(-1, 0)) * id);
        const double dtyx = (tyxp - tyxm) * id;
        const double tyyp = 2.0 * M(0, 1) * (V(0, 1) - V(0, 0)) * id;
        const double tyym = 2.0 * M(0, 0) * (V(0, 0) - V(0, -1)) * id;
        const double dtyy = (tyyp - tyym) * id;
        ry = ry + (dtyx + dtyy) / rfy;
    }
    // surface tension (CSF)
    {
        const double *K = a.curv + g, *F = a.vof + g;
        rx = rx + a.sigma * 0.5 * (K[1] + K[0]) * (F[1] - F[0]) * id / rfx;
        ry = ry + a.sigma * 0.5 * (K[sj] + K[0]) * (F[sj] - F[0]) * id / rfy;
    }
    if constexpr (SRC) {
        rx = rx + a.s0[q] / rfx;
        ry = ry + a.s1[q] / rfy;
    }
    const double p0 = a.p[g], ph0 = a.p_hat[g];
    {
        const double gp = (a.p[g + 1] - p0) * id, gh = (a.p_hat[g + 1] - ph0) * id;
        double rhs = ((-(gp / rfx) + a.A * rx) + a.B * a.dvo0[q]) + a.g0;
        rhs = ((rhs + gp / rfx) - a.irhomin * gp) - (1.0 / rfx - a.irhomin) * gh;
        const double val = u0 + a.dt * rhs;
        put_ghosted(a.gu, a.b, a.us, i, j, val);
        a.dvo0[q] = rx;
    }
    {
        const double gp = (a.p[g + sj] - p0) * id, gh = (a.p_hat[g + sj] - ph0) * id;
        double rhs = ((-(gp / rfy) + a.A * ry) + a.B * a.dvo1[q]) + a.g1;
        rhs = ((rhs + gp / rfy) - a.irhomin * gp) - (1.0 / rfy - a.irhomin) * gh;
        const double val = v0 + a.dt * rhs;
        put_ghosted(a.gv, a.b, a.vs, i, j, val);
        a.dvo1[q] = ry;
    }
}

dim3 cell_grid(const Box &b) { return dim3((unsigned)((b.nx + kBX - 1) / kBX), (unsigned)((b.ny + kBY - 1) / kBY)); }

MFCopies mf_copies(const fen_ctx *c)
{
    MFCopies m{};
    for (int f = 0; f < 4; f++) m.face[f] = c->bc_phys[f] == FEN_BC_PERIODIC ? COPY_PERIODIC : COPY_MIRROR;
    return m;
}

void vof_reconstruct(fen_ctx *c, const double *vof)
{
    MFState &m = *c->mf;
    VofArgs a{};
    a.copies = mf_copies(c);
    a.b = c->box;
    a.delta = c->delta;
    a.id = 1.0 / c->delta;
    a.id2 = 1.0 / (c->delta * c->delta);
    a.beta = m.beta;
    a.vof = vof;
    a.dd = m.dd; a.curv = m.curv; a.nrx = m.nrx; a.nry = m.nry; a.lx = m.lx; a.ly = m.ly;
    hipLaunchKernelGGL(vof_reconstruct_kernel, cell_grid(c->box), dim3(kBX * kBY), 0, c->stream, a);
}

SweepArgs sweep_args(fen_ctx *c, const double *vof, double *out, double dt)
{
    MFState &m = *c->mf;
    SweepArgs a{};
    a.copies = mf_copies(c);
    a.b = c->box;
    a.delta = c->delta;
    a.beta = m.beta;
    a.dt = dt;
    a.vof = vof; a.dd = m.dd; a.nrx = m.nrx; a.nry = m.nry; a.lx = m.lx; a.ly = m.ly;
    a.u = as<double>(c->d_u[0]);
    a.v = as<double>(c->d_u[1]);
    a.out = out;
    return a;
}

template <int DIR, int SECOND> void vof_sweep(fen_ctx *c, const SweepArgs &a)
{
    hipLaunchKernelGGL((vof_sweep_kernel<DIR, SECOND>), cell_grid(c->box), dim3(kFaces), 0, c->stream, a);
}

}  // namespace

void mf_ghost_field(fen_ctx *c, double *f)
{
    GhostDesc<double> d{};
    d.f = f;
    for (int face = 0; face < 4; face++) d.type[face] = c->bc_phys[face] == FEN_BC_PERIODIC ? 0 : 2;
    d.loc = 'c';
    d.groups = 3;
    launch_ghost_desc<double>(c, &d, 1);
}

// advect_vof (src/volume_of_fluid.f90:420-544) with the resident velocity;
// `fields`: also the material properties and p_hat (mf_update_fields).
void mf_advect_vof(fen_ctx *c, double dt, bool fields, double dt_hat)
{
    MFState &m = *c->mf;
    vof_reconstruct(c, m.vof);
    SweepArgs a = sweep_args(c, m.vof, m.vof1, dt);
    if (m.x_first) vof_sweep<1, 0>(c, a);
    else vof_sweep<2, 0>(c, a);
    vof_reconstruct(c, m.vof1);
    a = sweep_args(c, m.vof1, m.vof, dt);
    if (fields) {
        a.rho0 = m.rho0; a.rho1 = m.rho1; a.mu0 = m.mu0; a.mu1 = m.mu1;
        a.dt_hat = dt_hat;
        a.dt_o = c->dt_o;
        a.p = as<double>(c->d_p);
        a.p_o = m.p_o;
        a.rho = m.rho; a.mu = m.mu; a.p_hat = m.p_hat;
    }
    if (m.x_first) vof_sweep<2, 1>(c, a);
    else vof_sweep<1, 1>(c, a);
    m.x_first = !m.x_first;
}

// update_material_properties.
void mf_update_fields(fen_ctx *c)
{
    MFState &m = *c->mf;
    hipLaunchKernelGGL(mf_fields_kernel, cell_grid(c->box), dim3(kBX * kBY), 0, c->stream, c->box, mf_copies(c),
                       (const double *)m.vof, m.rho0, m.rho1, m.mu0, m.mu1, m.rho, m.mu);
}

void mf_momentum(fen_ctx *c, double dt)
{
    MFState &m = *c->mf;
    MFMomArgs a{};
    a.b = c->box;
    a.id = 1.0 / c->delta;
    a.dt = dt;
    a.A = 1.0 + 0.5 * dt / c->dt_o;   // src/navier_stokes.f90:157-158
    a.B = -(0.5 * dt / c->dt_o);
    a.g0 = c->g[0];
    a.g1 = c->g[1];
    a.sigma = m.sigma;
    a.irhomin = m.irhomin;
    a.u = as<double>(c->d_u[0]); a.v = as<double>(c->d_u[1]); a.p = as<double>(c->d_p);
    a.p_hat = m.p_hat; a.rho = m.rho; a.mu = m.mu; a.vof = m.vof; a.curv = m.curv;
    a.s0 = as<double>(c->d_S[0]); a.s1 = as<double>(c->d_S[1]);
    a.us = as<double>(c->d_us[0]); a.vs = as<double>(c->d_us[1]);
    a.dvo0 = as<double>(c->d_dvo[0]); a.dvo1 = as<double>(c->d_dvo[1]);
    a.gu = make_desc<double>(c, FEN_U, a.us);
    a.gv = make_desc<double>(c, FEN_V, a.vs);
    prof_begin(c, K_MOMENTUM);
    if (c->has_source) hipLaunchKernelGGL(mf_momentum_kernel<1>, cell_grid(c->box), dim3(kBX * kBY), 0, c->stream, a);
    else hipLaunchKernelGGL(mf_momentum_kernel<0>, cell_grid(c->box), dim3(kBX * kBY), 0, c->stream, a);
    prof_end(c, K_MOMENTUM, 8.0 * 16.0 * c->n_int);
}

}  // namespace fen
