// stencil_kernels.hip -- staggered-grid kernels of the time step, for field
// element type R = double (FP64) and R = float (the FP32 form).
//
// Every expression keeps the reference's evaluation order (Fortran left to
// right, explicit parentheses) and the library is compiled with
// -ffp-contract=off, so the FP64 kernels reproduce the CPU arithmetic bit
// for bit.
//
// Producers (momentum, projection) write the periodic images of the boundary
// cells they compute, so a periodic ghost fill costs no extra pass; the ghost
// kernel then runs only over the axes that are not periodic.
#include <algorithm>
#include <cmath>
#include <stdexcept>
#include <type_traits>

#include "fen_internal.hpp"
#include "stencil_march.hpp"

namespace fen {

constexpr int kTX = 64, kTY = 4, kThreads = kTX * kTY;

// ---------------------------------------------------------------------------
// Ghost fill: scalar%update_ghost_nodes (src/scalar.f90:223-396) evaluated
// as a pure function of the interior.  The reference fills left, right,
// bottom, top, front, back over full planes, so a ghost's final value is the
// last axis rule applied to the state left by the earlier axes:
//   S1 = x rules on the interior S0, S2 = y rules on S1, S3 = z rules on S2.
// A Dirichlet rule on a field's normal face at the high end also overwrites
// the last interior plane (f(N) = bc).  Every cell written here is computed
// from interior cells that no thread writes, so one launch needs no ordering.
// ---------------------------------------------------------------------------
constexpr int kGhostFields = 8;   // fields per ghost-fill launch
template <class R> struct GhostLaunch {
    GhostDesc<R> d[kGhostFields];
    Box b;
    int nx_cells, ny_cells, nz_cells;              // cells per plane of each group
    int ngx[kGhostFields], ngy[kGhostFields], ngz[kGhostFields];   // planes per group and field (0: skipped)
};

// The rules as one chain: the interior cell they start from (x, y and z apart),
// then what each axis makes of its value.  Straight-line code: as nested calls,
// inlined at each of their uses for each field, the kernel spent most of its
// time fetching instructions (u*, v*, w* at 128 x 128 x 160: 7.4 us; as one
// chain and on their normal faces only, 5.3).
template <class R> __device__ __forceinline__ R ghost_value(const GhostDesc<R> &d, const Box &b, int i, int j, int k)
{
    const R two = R(2.0);
    auto from = [](int g, int n, int lo, int hi) {
        return g == 0 ? (lo == 0 ? n : 1) : (g == n + 1 ? (hi == 0 ? 1 : n) : g);
    };
    const bool z = b.dim == 3;
    const int ix = from(i, b.nx, d.type[0], d.type[1]), jy = from(j, b.ny, d.type[2], d.type[3]);
    const int kz = z ? from(k, b.nz, d.type[4], d.type[5]) : k;
    R v = d.f[b.g(ix, jy, kz)];
    auto rule = [&](int g, int n, int face, char loc, long at) {
        const bool normal = d.loc == loc;
        const int t = g == 0 ? d.type[face] : (g == n + 1 || (g == n && normal) ? d.type[face + 1] : 0);
        if (t != 1) return;
        const R bc = g == 0 ? d.plane[face][at] : d.plane[face + 1][at];
        v = normal ? bc : two * bc - v;
    };
    rule(i, b.nx, 0, 'x', jy + (long)(b.ny + 2) * kz);
    rule(j, b.ny, 2, 'y', i + (long)(b.nx + 2) * kz);
    if (z) rule(k, b.nz, 4, 'z', i + (long)(b.nx + 2) * j);
    return v;
}

// Group plane index p -> coordinate: 0 -> 0, 1 -> n+1, 2 -> n (normal overwrite).
__device__ __forceinline__ int plane_coord(int p, int n) { return p == 0 ? 0 : (p == 1 ? n + 1 : n); }

// One field per blockIdx.y.  The descriptor is selected with a compile-time
// index (Q) and the rule functions above are inlined: a run-time index into
// the by-value argument block, or its address passed to a call that is not
// inlined, makes the compiler copy the whole block (464 bytes) into per-lane
// scratch memory, which cost 55 us per field at 256^3.
template <class R, int Q> __device__ __forceinline__ void ghost_field(const GhostLaunch<R> &a)
{
    const GhostDesc<R> &d = a.d[Q];
    const Box &b = a.b;
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int tx = a.nx_cells * a.ngx[Q], ty = a.ny_cells * a.ngy[Q], tz = a.nz_cells * a.ngz[Q];
    int i, j, k;
    if (t < tx) {
        // x faces: i ghost (or the overwritten normal plane), j and k interior
        const int p = t / a.nx_cells, r = t - p * a.nx_cells;
        i = plane_coord(p, b.nx);
        k = r / b.ny;
        j = r - k * b.ny + 1;
        k += 1;
    } else if ((t -= tx) < ty) {
        // y faces: j ghost, every i, k interior
        const int p = t / a.ny_cells, r = t - p * a.ny_cells;
        j = plane_coord(p, b.ny);
        k = r / (b.nx + 2);
        i = r - k * (b.nx + 2);
        k += 1;
    } else if ((t -= ty) < tz) {
        // z faces: k ghost, every i and j
        const int p = t / a.nz_cells, r = t - p * a.nz_cells;
        k = plane_coord(p, b.nz);
        j = r / (b.nx + 2);
        i = r - j * (b.nx + 2);
    } else {
        return;
    }
    d.f[b.g(i, j, k)] = ghost_value(d, b, i, j, k);
}

template <class R> __global__ __launch_bounds__(256) void ghost_kernel(GhostLaunch<R> a)
{
    switch (blockIdx.y) {
    case 0: ghost_field<R, 0>(a); break;
    case 1: ghost_field<R, 1>(a); break;
    case 2: ghost_field<R, 2>(a); break;
    case 3: ghost_field<R, 3>(a); break;
    case 4: ghost_field<R, 4>(a); break;
    case 5: ghost_field<R, 5>(a); break;
    case 6: ghost_field<R, 6>(a); break;
    default: ghost_field<R, 7>(a); break;
    }
}

template <class R> void launch_ghost_desc(fen_ctx *c, const GhostDesc<R> *descs, int n)
{
    if (n <= 0 || n > kGhostFields) throw std::runtime_error("ghost fill of 1..8 fields");
    GhostLaunch<R> a{};
    const Box &b = c->box;
    a.b = b;
    a.nx_cells = b.ny * b.nz;
    a.ny_cells = (b.nx + 2) * b.nz;
    a.nz_cells = (b.nx + 2) * (b.ny + 2);
    long most = 0;
    double cells = 0.0;
    for (int q = 0; q < n; q++) {
        const GhostDesc<R> &d = descs[q];
        a.d[q] = d;
        a.ngx[q] = (d.groups & 1) ? (d.type[FEN_RIGHT] == 1 && d.loc == 'x' ? 3 : 2) : 0;
        a.ngy[q] = (d.groups & 2) ? (d.type[FEN_TOP] == 1 && d.loc == 'y' ? 3 : 2) : 0;
        a.ngz[q] = (b.dim == 3 && (d.groups & 4)) ? (d.type[FEN_BACK] == 1 && d.loc == 'z' ? 3 : 2) : 0;
        const long tot = (long)a.nx_cells * a.ngx[q] + (long)a.ny_cells * a.ngy[q] + (long)a.nz_cells * a.ngz[q];
        most = tot > most ? tot : most;
        cells += (double)tot;
    }
    if (most == 0) return;
    if (most > INT32_MAX - 256) throw std::runtime_error("ghost fill: too many cells for 32-bit indices");
    const dim3 grid((unsigned)((most + 255) / 256), (unsigned)n);
    prof_begin(c, K_GHOST);
    hipLaunchKernelGGL(ghost_kernel<R>, grid, dim3(256), 0, c->stream, a);
    prof_end(c, K_GHOST, 2.0 * sizeof(R) * cells);
}

// The mean of phi from its block sums (n <= 256), by mean_shift_kernel's own
// tree, in every wave by itself: no barrier.
__device__ __forceinline__ double wave_mean(const double *part, int n, double count)
{
    const int l = threadIdx.x & 63;
    auto at = [&](int q) { return q < n ? part[q] : 0.0; };
    double x = (at(l) + at(l + 128)) + (at(l + 64) + at(l + 192));
    for (int s = 32; s > 0; s >>= 1) x = x + __shfl_down(x, s);
    return __shfl(x, 0) / count;
}

// 2-D: one cell per thread, neighbours straight from memory (the whole
// 128^2 problem fits in cache); u* and v* are left with their ghosts filled.
template <class R> struct Ghosts2D {
    GhostDesc<R> d[3];
};
template <class R, int SRC>
__global__ __launch_bounds__(kThreads) void momentum_kernel_2d(MomArgs<R> a, Ghosts2D<R> gh)
{
    const int i = blockIdx.x * kTX + (threadIdx.x % kTX) + 1;
    const int j = blockIdx.y * kTY + (threadIdx.x / kTX) + 1;
    if (i > a.b.nx || j > a.b.ny) return;
    const long g = a.b.g(i, j, 1), sj = a.b.gx;
    auto at = [&](const R *f) {
        return [=](int di, int dj, int dk) { return f[g + di + sj * dj]; };
    };
    const long q = a.b.q(i, j, 1);
    R val[2] = {R(0), R(0)};
    auto keep = [&](R *f, R v) { (f == a.us ? val[0] : val[1]) = v; };
    momentum_cell<0, SRC>(a, i, j, 1, at(a.u), at(a.v), at(a.w), at(a.p), a.dvo0[q], a.dvo1[q], R(0), keep);
    put_ghosted(gh.d[0], a.b, a.us, i, j, val[0]);
    put_ghosted(gh.d[1], a.b, a.vs, i, j, val[1]);
}

// 3-D launch shapes (see stencil_march.hpp), chosen per element type by a
// sweep of tile height, planes per workgroup, ring unrolling and prefetch
// depth on MI355X at 256^3.
// (tile height TY, planes per workgroup KB, ring unrolling UN, prefetch depth
// PF, minimum waves per SIMD for the register allocation OCC.  128-wide
// momentum and projection tiles gained 0.6% on the per-step path of the
// Neumann solvers and are not used: MTXW = PTXW = 64)
template <class R> struct Shape;
template <> struct Shape<double> {
    static constexpr int MTY = 8, MKB = 32, MUN = 1, MPF = 1, MOCC = 1, MTXW = 64;   // momentum
    static constexpr int PTY = 4, PKB = 16, PUN = 1, PPF = 1, POCC = 1, PTXW = 64;   // projection
};
template <> struct Shape<float> {
    static constexpr int MTY = 4, MKB = 16, MUN = 2, MPF = 2, MOCC = 1, MTXW = 64;
    static constexpr int PTY = 4, PKB = 16, PUN = 1, PPF = 1, POCC = 4, PTXW = 64;
};
constexpr int MTX = 64;

static void grid_blocks(const Box &b, int ty, int kb, int *nbx, int *nby, int *nbz, int tx = MTX)
{
    if (b.dim == 3) {
        *nbx = (b.nx + tx - 1) / tx;
        *nby = (b.ny + ty - 1) / ty;
        *nbz = (b.nz + kb - 1) / kb;
    } else {
        *nbx = (b.nx + kTX - 1) / kTX;
        *nby = (b.ny + kTY - 1) / kTY;
        *nbz = 1;
    }
}

// Workgroups of project_checks_kernel, each marching kb planes of 64 x 8 cells.
constexpr int kCheckPlanes = 8;
static long checks_blocks(const Box &b, int kb)
{
    return (long)((b.nx + 63) / 64) * ((b.ny + 7) / 8) * (b.dim == 3 ? (b.nz + kb - 1) / kb : 1);
}

// Workgroups of the kernels that write one partial each (the projection),
// either element type: the partial buffer's size.
long stencil_blocks(const Box &b)
{
    const int shapes[2][3] = {{Shape<double>::PTY, Shape<double>::PKB, Shape<double>::PTXW},
                              {Shape<float>::PTY, Shape<float>::PKB, Shape<float>::PTXW}};
    long most = 0;
    for (const auto &sh : shapes) {
        int nbx, nby, nbz;
        grid_blocks(b, sh[0], sh[1], &nbx, &nby, &nbz, sh[2]);
        most = std::max(most, (long)nbx * nby * nbz);
    }
    return std::max(most, checks_blocks(b, kCheckPlanes));
}

template <class R> void launch_momentum(fen_ctx *c, double dt, double A, double B)
{
    MomArgs<R> a = momentum_args<R>(c, dt, A, B);
    int nbz;
    using SH = Shape<R>;
    grid_blocks(c->box, SH::MTY, SH::MKB, &a.nbx, &a.nby, &nbz, SH::MTXW);
    const int d3 = c->box.dim == 3;
    const double words = d3 ? (c->has_source ? 16.0 : 13.0) : (c->has_source ? 11.0 : 9.0);
    prof_begin(c, K_MOMENTUM);
    if (d3) {
        const dim3 grid((unsigned)(a.nbx * a.nby * nbz));
        if (c->has_source)
            hipLaunchKernelGGL((momentum_march_kernel<R, 1, SH::MTY, SH::MKB, SH::MUN, SH::MPF, SH::MOCC, SH::MTXW>),
                               grid, dim3(SH::MTXW * SH::MTY), 0, c->stream, a);
        else
            hipLaunchKernelGGL((momentum_march_kernel<R, 0, SH::MTY, SH::MKB, SH::MUN, SH::MPF, SH::MOCC, SH::MTXW>),
                               grid, dim3(SH::MTXW * SH::MTY), 0, c->stream, a);
    } else {
        const dim3 grid((unsigned)a.nbx, (unsigned)a.nby);
        Ghosts2D<R> gh{};
        gh.d[0] = make_desc<R>(c, FEN_U, a.us);
        gh.d[1] = make_desc<R>(c, FEN_V, a.vs);
        if (c->has_source) hipLaunchKernelGGL((momentum_kernel_2d<R, 1>), grid, dim3(kThreads), 0, c->stream, a, gh);
        else hipLaunchKernelGGL((momentum_kernel_2d<R, 0>), grid, dim3(kThreads), 0, c->stream, a, gh);
    }
    prof_end(c, K_MOMENTUM, words * sizeof(R) * c->n_int);
}

// add_advection alone on the resident velocity (reference test
// test/small_test/navier_stokes/advection/advection.f90:50): R -= adv.
template <int D3>
__global__ __launch_bounds__(kThreads) void advection_kernel(const double *u, const double *v, const double *w,
                                                             double *rx, double *ry, double *rz, Box b, double id)
{
    const int i = blockIdx.x * kTX + (threadIdx.x % kTX) + 1;
    const int j = blockIdx.y * kTY + (threadIdx.x / kTX) + 1;
    const int k = D3 ? (int)blockIdx.z + 1 : 1;
    if (i > b.nx || j > b.ny) return;
    const long g = b.g(i, j, k), q = b.q(i, j, k);
    const long sj = b.gx, sk = b.gxy;
    const double *U = u + g, *V = v + g, *W = w + g;
    double uuip = 0.25 * ((U[1] + U[0]) * (U[1] + U[0]));
    double uuim = 0.25 * ((U[-1] + U[0]) * (U[-1] + U[0]));
    double uvjp = ((U[sj] + U[0]) * (V[1] + V[0])) * 0.25;
    double uvjm = ((U[0] + U[-sj]) * (V[1 - sj] + V[-sj])) * 0.25;
    double r = (rx[q] - (uuip - uuim) * id) - (uvjp - uvjm) * id;
    if constexpr (D3) {
        double uwkp = ((U[sk] + U[0]) * (W[1] + W[0])) * 0.25;
        double uwkm = ((U[0] + U[-sk]) * (W[1 - sk] + W[-sk])) * 0.25;
        r = r - (uwkp - uwkm) * id;
    }
    rx[q] = r;
    double vuip = ((V[1] + V[0]) * (U[sj] + U[0])) * 0.25;
    double vuim = ((V[0] + V[-1]) * (U[-1 + sj] + U[-1])) * 0.25;
    double vvjp = 0.25 * ((V[sj] + V[0]) * (V[sj] + V[0]));
    double vvjm = 0.25 * ((V[-sj] + V[0]) * (V[-sj] + V[0]));
    r = (ry[q] - (vuip - vuim) * id) - (vvjp - vvjm) * id;
    if constexpr (D3) {
        double vwkp = ((V[sk] + V[0]) * (W[sj] + W[0])) * 0.25;
        double vwkm = ((V[0] + V[-sk]) * (W[sj - sk] + W[-sk])) * 0.25;
        r = r - (vwkp - vwkm) * id;
    }
    ry[q] = r;
    if constexpr (D3) {
        double wuip = ((W[0] + W[1]) * (U[0] + U[sk])) * 0.25;
        double wuim = ((W[0] + W[-1]) * (U[-1] + U[-1 + sk])) * 0.25;
        double wvjp = ((W[0] + W[sj]) * (V[0] + V[sk])) * 0.25;
        double wvjm = ((W[0] + W[-sj]) * (V[-sj] + V[-sj + sk])) * 0.25;
        double wwkp = ((W[0] + W[sk]) * (W[0] + W[sk])) * 0.25;
        double wwkm = ((W[0] + W[-sk]) * (W[0] + W[-sk])) * 0.25;
        rz[q] = ((rz[q] - (wuip - wuim) * id) - (wvjp - wvjm) * id) - (wwkp - wwkm) * id;
    }
}

void launch_advection_only(fen_ctx *c, double *rx, double *ry, double *rz)
{
    const Box &b = c->box;
    const dim3 grid((unsigned)((b.nx + kTX - 1) / kTX), (unsigned)((b.ny + kTY - 1) / kTY),
                    (unsigned)(b.dim == 3 ? b.nz : 1));
    const double *u = as<double>(c->d_u[0]), *v = as<double>(c->d_u[1]), *w = as<double>(c->d_u[2]);
    if (b.dim == 3)
        hipLaunchKernelGGL((advection_kernel<1>), grid, dim3(kThreads), 0, c->stream, u, v, w, rx, ry, rz, b,
                           1.0 / c->delta);
    else
        hipLaunchKernelGGL((advection_kernel<0>), grid, dim3(kThreads), 0, c->stream, u, v, w, rx, ry, rz, b,
                           1.0 / c->delta);
}

// The projection, pressure update and checks of a 2-D step, u, v and p left
// with their ghosts filled.  nparts > 0: the mean of phi is still in its block
// sums and every workgroup adds them (a launch of its own took 4 us).  p_old:
// receives p before the update (two-phase).  ST == 0: the checks only.
template <class R> struct Project2D {
    Ghosts2D<R> gh;   // u, v, p
    const double *part;
    double count;
    int nparts;
    R *p_old;
};
template <class R, int SHIFT, int ST>
__global__ __launch_bounds__(kThreads) void project_kernel_2d(ProjArgs<R> a, Project2D<R> x)
{
    const int i = blockIdx.x * kTX + (threadIdx.x % kTX) + 1;
    const int j = blockIdx.y * kTY + (threadIdx.x / kTX) + 1;
    const Box &b = a.b;
    double md = -HUGE_VAL, mv = 0.0, bad = 0.0;
    double s = 0.0;
    if constexpr (SHIFT) s = x.nparts > 0 ? wave_mean(x.part, x.nparts, x.count) : a.shift[0];
    if (i <= b.nx && j <= b.ny) {
        const long g = b.g(i, j, 1), sj = b.gx;
        auto F = [&](int di, int dj, int dk) -> double {
            if constexpr (SHIFT) return (double)a.phi[g + di + sj * dj] - s;
            else return (double)a.phi[g + di + sj * dj];
        };
        R val[3] = {R(0), R(0), R(0)};
        auto keep = [&](R *f, R v) { (f == a.u ? val[0] : (f == a.v ? val[1] : val[2])) = v; };
        const R p0 = ST ? a.p[g] : R(0);
        project_cell<0, R, decltype(F), decltype(keep), ST>(a, i, j, 1, F, a.us[g], a.vs[g], 0.0, p0, a.us[g - 1],
                                                            a.vs[g - sj], 0.0, md, mv, bad, keep);
        if constexpr (ST) {
            if (x.p_old) x.p_old[g] = p0;
            put_ghosted(x.gh.d[0], b, a.u, i, j, val[0]);
            put_ghosted(x.gh.d[1], b, a.v, i, j, val[1]);
            put_ghosted(x.gh.d[2], b, a.p, i, j, val[2]);
        }
    }
    block_max3<kThreads>(md, mv, bad, a.part, (long)blockIdx.y * gridDim.x + blockIdx.x);
}

// One workgroup reduces the per-workgroup partials and leaves the maxima in
// out, pinned host memory: a reader waits for this kernel instead of queueing
// a copy behind it.  Each thread issues the loads of B entries before comparing
// any, so the pass costs about one memory latency per B entries instead of one
// per entry.
constexpr int kFinalThreads = 1024;
__global__ __launch_bounds__(kFinalThreads) void checks_final_kernel(const double *part, long n, double *out)
{
    constexpr int NT = kFinalThreads, B = 4;
    double md = -HUGE_VAL, mv = 0.0, bad = 0.0;
    for (long q0 = threadIdx.x; q0 < n; q0 += (long)NT * B) {
        double x[B][3];
#pragma unroll
        for (int m = 0; m < B; m++) {
            const long q = q0 + (long)m * NT;
            const long qq = q < n ? q : q0;   // a valid entry; its value is dropped below
            x[m][0] = part[3 * qq];
            x[m][1] = part[3 * qq + 1];
            x[m][2] = part[3 * qq + 2];
        }
#pragma unroll
        for (int m = 0; m < B; m++) {
            if (q0 + (long)m * NT >= n) continue;
            if (x[m][0] > md) md = x[m][0];
            if (x[m][1] > mv) mv = x[m][1];
            if (x[m][2] > bad) bad = x[m][2];
        }
    }
    block_max3<NT>(md, mv, bad, out, 0);
}

// Step n's projection and pressure update fused with step n+1's momentum in
// 2-D: the state of step n is formed in LDS for a 64 x 4 tile and its halo (the
// projection of the interior cell the ghost fill reads, then the fill's rule
// chain on a wall position), p of step n is stored and the tile advanced to u*,
// v* of step n+1, left with their ghosts filled.  Latency bounds it, as every
// 2-D kernel: the projection (6.9 us at 128^2) and momentum (4.1) apart, one
// launch of 5.5 together.
template <class R> struct Step2D {
    MomArgs<R> m;                            // momentum of step n+1 (m.u, m.v, m.p unused)
    Ghosts2D<R> gh;                          // its u*, v*
    const R *us, *vs, *phi, *p_in;           // step n
    R *p_out;
    const double *shift, *part;              // pending mean of phi, or its block sums (nparts > 0)
    double count;
    int nparts;
    double id, dt, rhof, irhof;
    int rpow2;
    int wall, gtype[3];                      // PMArgs::wall, gtype of u, v, p
    const R *const *gplane;                  // PMArgs::gplane (u, v, w, p)
};
template <class R, int SRC, int SHIFT>
__global__ __launch_bounds__(kThreads) void step_kernel_2d(Step2D<R> a)
{
    constexpr int LX = kTX + 2, N = LX * (kTY + 2), PER = (N + kThreads - 1) / kThreads;
    __shared__ R lds[3][N];
    const Box &b = a.m.b;
    const int i0 = blockIdx.x * kTX + 1, j0 = blockIdx.y * kTY + 1;
    // every load is issued before the mean is known
    R raw[PER][6];
    int gi[PER], gj[PER];
#pragma unroll
    for (int q = 0; q < PER; q++) {
        const int e = threadIdx.x + q * kThreads, ee = e < N ? e : 0;
        gi[q] = min(i0 - 1 + ee % LX, b.nx + 1);
        gj[q] = min(j0 - 1 + ee / LX, b.ny + 1);
        const long o = b.g(pm_src(gi[q], b.nx, a.wall & 1), pm_src(gj[q], b.ny, a.wall & 2), 1);
        raw[q][0] = a.us[o];
        raw[q][1] = a.vs[o];
        raw[q][2] = a.p_in[o];
        raw[q][3] = a.phi[o];
        raw[q][4] = a.phi[o + 1];
        raw[q][5] = a.phi[o + b.gx];
    }
    double s = 0.0;
    if constexpr (SHIFT) s = a.nparts > 0 ? wave_mean(a.part, a.nparts, a.count) : a.shift[0];
    auto dr = [&](double x) { return over_rho(x, a.rhof, a.irhof, a.rpow2); };
#pragma unroll
    for (int q = 0; q < PER; q++) {
        const int e = threadIdx.x + q * kThreads;
        double f0 = (double)raw[q][3], fx = (double)raw[q][4], fy = (double)raw[q][5];
        if constexpr (SHIFT) {
            f0 = f0 - s; fx = fx - s; fy = fy - s;
        }
        R st[3] = {(R)((double)raw[q][0] - dr((fx - f0) * a.id * a.dt)), (R)((double)raw[q][1] - dr((fy - f0) * a.id * a.dt)),
                   (R)((double)raw[q][2] + f0)};
        if (((a.wall & 1) && pm_wall_pos(gi[q], b.nx) >= 0) || ((a.wall & 2) && pm_wall_pos(gj[q], b.ny) >= 0)) {
            const int jy = pm_src(gj[q], b.ny, a.wall & 2);
#pragma unroll
            for (int f = 0; f < 3; f++)
                st[f] = pm_ghost_chain(a.gtype[f], a.gplane + 6 * (f == 2 ? 3 : f), b, a.wall & 3, gi[q], gj[q], 1, jy, 1, st[f]);
        }
        if (e < N)
#pragma unroll
            for (int f = 0; f < 3; f++) lds[f][e] = st[f];
    }
    __syncthreads();
    const int tx = threadIdx.x % kTX, ty = threadIdx.x / kTX, i = i0 + tx, j = j0 + ty;
    if (i > b.nx || j > b.ny) return;
    const int c = (ty + 1) * LX + tx + 1;
    auto at = [&](int f) {
        return [=](int di, int dj, int dk) { return lds[f][c + dj * LX + di]; };
    };
    const long q = b.q(i, j, 1);
    a.p_out[b.g(i, j, 1)] = lds[2][c];
    R val[2] = {R(0), R(0)};
    auto keep = [&](R *f, R v) { (f == a.m.us ? val[0] : val[1]) = v; };
    momentum_cell<0, SRC>(a.m, i, j, 1, at(0), at(1), at(0), at(2), a.m.dvo0[q], a.m.dvo1[q], R(0), keep);
    put_ghosted(a.gh.d[0], b, a.m.us, i, j, val[0]);
    put_ghosted(a.gh.d[1], b, a.m.vs, i, j, val[1]);
}

// Whether a 2-D step may end with its projection pending: every axis of u, v,
// p and phi periodic on both faces, or walled on both (Dirichlet or Neumann);
// phi's walls Neumann (its ghosts are then filled by the solve).
bool fused_2d(const fen_ctx *c)
{
    if (c->box.dim != 2) return false;
    for (int ax = 0; ax < 2; ax++)
        for (int f : {FEN_U, FEN_V, FEN_P, FEN_PHI})
            for (int side = 0; side < 2; side++) {
                const int t = c->bc_type[f][2 * ax + side];
                if (c->periodic[ax] ? t != 0 : (f == FEN_PHI ? t != 2 : t != 1 && t != 2)) return false;
            }
    return true;
}

// us_in, p_in: u*, v* and p of step n; us_out, p_out: u*, v* of step n+1 and p
// after step n (distinct arrays).
template <class R>
void launch_step_2d(fen_ctx *c, double dt_p, double dt_m, double A, double B, void *const *us_in, const void *p_in,
                    void *const *us_out, void *p_out)
{
    if (!fused_2d(c)) throw std::runtime_error("fused 2-D step needs periodic or walled axes");
    Step2D<R> a{};
    a.m = momentum_args<R>(c, dt_m, A, B);
    a.m.us = as<R>(us_out[0]);
    a.m.vs = as<R>(us_out[1]);
    a.gh.d[0] = make_desc<R>(c, FEN_U, a.m.us);
    a.gh.d[1] = make_desc<R>(c, FEN_V, a.m.vs);
    a.us = as<R>(us_in[0]);
    a.vs = as<R>(us_in[1]);
    a.phi = as<R>(c->d_phi);
    a.p_in = static_cast<const R *>(p_in);
    a.p_out = as<R>(p_out);
    a.shift = c->d_shift;
    a.part = c->d_part;
    a.nparts = (int)c->shift_parts;
    a.count = (double)(float)((long)c->nx * c->ny * c->nz);
    a.id = 1.0 / c->delta;
    a.dt = dt_p;
    a.rhof = 0.5 * (c->density + c->density);
    a.rpow2 = pow2_value(a.rhof) ? 1 : 0;
    a.irhof = a.rpow2 ? 1.0 / a.rhof : 0.0;
    a.wall = (c->periodic[0] ? 0 : 1) | (c->periodic[1] ? 0 : 2);
    const int fid[3] = {FEN_U, FEN_V, FEN_P}, loc[3] = {1, 2, 0};
    for (int q = 0; q < 3; q++) {
        a.gtype[q] = loc[q] << 12;
        for (int f = 0; f < 4; f++) a.gtype[q] |= c->bc_type[fid[q]][f] << (2 * f);
    }
    a.gplane = reinterpret_cast<const R *const *>(c->d_plane_tab);
    const dim3 grid((unsigned)((c->nx + kTX - 1) / kTX), (unsigned)((c->ny + kTY - 1) / kTY));
    prof_begin(c, K_PROJ_MOM);
#define FEN_S2(SRC, SH) hipLaunchKernelGGL((step_kernel_2d<R, SRC, SH>), grid, dim3(kThreads), 0, c->stream, a)
    if (c->has_source) {
        if (c->shift_active) FEN_S2(1, 1);
        else FEN_S2(1, 0);
    } else {
        if (c->shift_active) FEN_S2(0, 1);
        else FEN_S2(0, 0);
    }
#undef FEN_S2
    // reads u*, v*, p, phi, dv_o (+ S); writes p, u*, v*, dv_o
    prof_end(c, K_PROJ_MOM, (c->has_source ? 13.0 : 11.0) * sizeof(R) * c->n_int);
}

void read_checks(fen_ctx *c)
{
    if (c->chk_blocks <= 0) return;
    prof_begin(c, K_REDUCE);
    hipLaunchKernelGGL(checks_final_kernel, dim3(1), dim3(kFinalThreads), 0, c->stream, (const double *)c->d_chk,
                       c->chk_blocks, c->h_scal);
    prof_end(c, K_REDUCE, 24.0 * c->chk_blocks);
    FEN_HIP_CHECK(hipGetLastError());
    FEN_HIP_CHECK(hipStreamSynchronize(c->stream));
    c->chk_blocks = 0;
}

template <class R> void launch_project(fen_ctx *c, double dt, bool store, R *p_old)
{
    if (p_old && c->box.dim != 2) throw std::runtime_error("the pressure before the step is kept in 2-D only");
    ProjArgs<R> a{};
    a.us = as<R>(c->d_us[0]); a.vs = as<R>(c->d_us[1]); a.ws = as<R>(c->d_us[2]); a.phi = as<R>(c->d_phi);
    a.u = as<R>(c->d_u[0]); a.v = as<R>(c->d_u[1]); a.w = as<R>(c->d_u[2]); a.p = as<R>(c->d_p);
    a.shift = c->d_shift;
    a.part = c->d_chk;
    const int lo[3] = {FEN_LEFT, FEN_BOTTOM, FEN_FRONT}, hi[3] = {FEN_RIGHT, FEN_TOP, FEN_BACK};
    for (int d = 0; d < 3; d++) {
        const int slot = FEN_U + d;
        a.lo_type[d] = c->bc_type[slot][lo[d]];
        a.hi_type[d] = c->bc_type[slot][hi[d]];
        a.lo_plane[d] = as<R>(c->d_plane[slot][lo[d]]);
        a.hi_plane[d] = as<R>(c->d_plane[slot][hi[d]]);
    }
    a.b = c->box;
    a.id = 1.0 / c->delta;
    a.dt = dt;
    a.rhof = 0.5 * (c->density + c->density);
    a.rpow2 = pow2_value(a.rhof) ? 1 : 0;
    a.irhof = a.rpow2 ? 1.0 / a.rhof : 0.0;
    if (c->mf) {   // MF: v - grad(phi) dt / rho_min as (grad(phi) dt) * irhomin (src/navier_stokes.f90:526-531)
        a.rhof = c->mf->rhomin;
        a.rpow2 = 1;
        a.irhof = c->mf->irhomin;
    }
    a.img = c->img_vel & c->img_p;
    int nbz;
    using SH = Shape<R>;
    grid_blocks(c->box, SH::PTY, SH::PKB, &a.nbx, &a.nby, &nbz, SH::PTXW);
    long nblk = (long)a.nbx * a.nby * nbz;
    const bool sh = c->shift_active;
    const int d3 = c->box.dim == 3;
    int kb = kCheckPlanes;
    if (d3 && !store) {
        // shorter marches (each loads two planes more) where they leave CUs idle
        while (kb > 2 && checks_blocks(c->box, kb) < 2L * c->num_cu && (size_t)(3 * checks_blocks(c->box, kb / 2)) <= c->n_chk)
            kb /= 2;
        a.nbx = (c->nx + 63) / 64;
        a.nby = (c->ny + 7) / 8;
        nblk = checks_blocks(c->box, kb);
    }
    if ((size_t)(3 * nblk) > c->n_chk) throw std::runtime_error("partial buffer too small");
    const int kid = store ? K_PROJECT : K_CHECKS;
    prof_begin(c, kid);
    if (d3 && !store) {
        if (sh) hipLaunchKernelGGL((project_checks_kernel<R, 1>), dim3((unsigned)nblk), dim3(256), 0, c->stream, a, kb);
        else hipLaunchKernelGGL((project_checks_kernel<R, 0>), dim3((unsigned)nblk), dim3(256), 0, c->stream, a, kb);
    } else if (d3) {
        const dim3 grid((unsigned)nblk);
#define FEN_PJ(SH_)                                                                                            \
    hipLaunchKernelGGL((project_march_kernel<R, SH_, SH::PTY, SH::PKB, SH::PUN, SH::PPF, SH::POCC, SH::PTXW>), \
                       grid, dim3(SH::PTXW * SH::PTY), 0, c->stream, a)
        if (sh) FEN_PJ(1);
        else FEN_PJ(0);
#undef FEN_PJ
    } else {
        const dim3 grid((unsigned)a.nbx, (unsigned)a.nby);
        Project2D<R> x{};
        x.gh.d[0] = make_desc<R>(c, FEN_U, a.u);
        x.gh.d[1] = make_desc<R>(c, FEN_V, a.v);
        x.gh.d[2] = make_desc<R>(c, FEN_P, a.p);
        x.part = c->d_part;
        x.nparts = (int)c->shift_parts;
        x.count = (double)(float)((long)c->nx * c->ny * c->nz);
        x.p_old = p_old;
#define FEN_PJ2(SH_, ST_) \
    hipLaunchKernelGGL((project_kernel_2d<R, SH_, ST_>), grid, dim3(kThreads), 0, c->stream, a, x)
        if (store) {
            if (sh) FEN_PJ2(1, 1);
            else FEN_PJ2(0, 1);
        } else {
            if (sh) FEN_PJ2(1, 0);
            else FEN_PJ2(0, 0);
        }
#undef FEN_PJ2
    }
    // the checks alone read u*, v*, w* and phi
    prof_end(c, kid, (store ? (d3 ? 9.0 : 7.0) : 4.0) * sizeof(R) * c->n_int);
    c->chk_blocks = nblk;
}

// ---------------------------------------------------------------------------
// Stand-alone checks on the resident velocity (used before the first step
// of a CFL-controlled run): same quantities as above, ghosts already filled.
// ---------------------------------------------------------------------------
constexpr int kCheckBlocks = 1024;

template <class R, int D3>
__global__ __launch_bounds__(256) void checks_kernel(const R *u, const R *v, const R *w, Box b, double id,
                                                     double *part)
{
    __shared__ double sd[256], sv[256], sf[256];
    const long n = (long)b.nx * b.ny * b.nz;
    double md = -HUGE_VAL, mv = 0.0, bad = 0.0;
    for (long t = (long)blockIdx.x * 256 + threadIdx.x; t < n; t += (long)gridDim.x * 256) {
        const int i = (int)(t % b.nx) + 1;
        const long r = t / b.nx;
        const int j = (int)(r % b.ny) + 1, k = (int)(r / b.ny) + 1;
        const long g = b.g(i, j, k);
        const double ug = u[g], vg = v[g];
        double d = (ug - (double)u[g - 1]) * id + (vg - (double)v[g - b.gx]) * id;
        if constexpr (D3) d = d + ((double)w[g] - (double)w[g - b.gxy]) * id;
        double vel = fabs(ug) + fabs(vg);
        if constexpr (D3) vel = vel + fabs((double)w[g]);
        if (!(d == d) || !(vel == vel) || isinf(vel)) bad = 1.0;
        if (d > md) md = d;
        if (vel > mv) mv = vel;
    }
    sd[threadIdx.x] = md; sv[threadIdx.x] = mv; sf[threadIdx.x] = bad;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            if (sd[threadIdx.x + s] > sd[threadIdx.x]) sd[threadIdx.x] = sd[threadIdx.x + s];
            if (sv[threadIdx.x + s] > sv[threadIdx.x]) sv[threadIdx.x] = sv[threadIdx.x + s];
            if (sf[threadIdx.x + s] > sf[threadIdx.x]) sf[threadIdx.x] = sf[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[3 * blockIdx.x + 0] = sd[0];
        part[3 * blockIdx.x + 1] = sv[0];
        part[3 * blockIdx.x + 2] = sf[0];
    }
}

template <class R> void launch_checks(fen_ctx *c, const R *const *vel)
{
    const Box &b = c->box;
    const double id = 1.0 / c->delta;
    long nblk = ((long)c->n_int + 255) / 256;
    if (nblk > kCheckBlocks) nblk = kCheckBlocks;
    if ((size_t)(3 * nblk) > c->n_chk) throw std::runtime_error("partial buffer too small");
    prof_begin(c, K_CHECKS);
    if (b.dim == 3)
        hipLaunchKernelGGL((checks_kernel<R, 1>), dim3((unsigned)nblk), dim3(256), 0, c->stream, vel[0], vel[1],
                           vel[2], b, id, c->d_chk);
    else
        hipLaunchKernelGGL((checks_kernel<R, 0>), dim3((unsigned)nblk), dim3(256), 0, c->stream, vel[0], vel[1],
                           vel[2], b, id, c->d_chk);
    prof_end(c, K_CHECKS, (b.dim == 3 ? 3.0 : 2.0) * sizeof(R) * c->n_int);
    c->chk_blocks = nblk;
}

template void launch_ghost_desc<double>(fen_ctx *, const GhostDesc<double> *, int);
template void launch_ghost_desc<float>(fen_ctx *, const GhostDesc<float> *, int);
template void launch_momentum<double>(fen_ctx *, double, double, double);
template void launch_momentum<float>(fen_ctx *, double, double, double);
template void launch_project<double>(fen_ctx *, double, bool, double *);
template void launch_project<float>(fen_ctx *, double, bool, float *);
template void launch_step_2d<double>(fen_ctx *, double, double, double, double, void *const *, const void *, void *const *,
                                     void *);
template void launch_step_2d<float>(fen_ctx *, double, double, double, double, void *const *, const void *, void *const *,
                                    void *);
template void launch_checks<double>(fen_ctx *, const double *const *);
template void launch_checks<float>(fen_ctx *, const float *const *);

}  // namespace fen
