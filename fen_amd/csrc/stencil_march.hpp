// stencil_march.hpp -- k-marching launch shape of the 3-D momentum and
// projection kernels.
//
// A workgroup owns a 64 x TY tile of (i, j) and marches KB planes in k.
// Planes k-1, k, k+1 of the stencil inputs, each with a one-cell halo in i
// and j, sit in a 3-slot LDS ring, so every value is read from HBM once per
// tile plus the halo.  The ring is software-pipelined: the global loads of
// plane k+2 are issued into registers before plane k is computed and are
// written to LDS one iteration later, so HBM latency overlaps arithmetic.
// Inputs needed only at the cell itself (dv_o; w*, p in the projection) are
// prefetched one plane ahead in registers.  With UNROLL == 3 the k loop is
// unrolled by three so every ring slot is a compile-time LDS offset.  With
// PF == 2 two register sets alternate, so planes k+2 and k+3 are in flight
// together (UNROLL == 2, ring slots at run time): twice the bytes in flight
// per wave, which FP32 fields need to cover the same HBM latency.
#pragma once

#include <type_traits>

#include "stencil_cells.hpp"

namespace fen {

// NJ: rows (adjacent in j) computed by one thread.
template <int TY, int TX_ = 64, int NJ = 1> struct TileShape {
    static_assert(TY % NJ == 0, "whole rows per thread");
    static constexpr int TX = TX_, LX = TX + 2, LY = TY + 2, N = LX * LY, NT = TX * TY / NJ;
    static constexpr int PER = (N + NT - 1) / NT;
};

// Per-thread tile elements.  Loads and LDS writes are unconditional: an
// element past the tile reads a valid address (the tile corner) and writes a
// scratch row after the ring, and halo cells past the grid are clamped onto
// it; neither is ever read by an active cell.
template <class S> struct TileIdx {
    int off[S::PER];   // element offset in the ghosted array at k = 0
};

template <class S> __device__ __forceinline__ TileIdx<S> tile_index(const Box &b, int i0, int j0)
{
    TileIdx<S> t;
#pragma unroll
    for (int q = 0; q < S::PER; q++) {
        const int e = threadIdx.x + q * S::NT;
        const int ri = e % S::LX, rj = e / S::LX;
        int gi = min(i0 - 1 + ri, b.nx + 1), gj = min(j0 - 1 + rj, b.ny + 1);
        if (e >= S::N) { gi = i0 - 1; gj = j0 - 1; }
        t.off[q] = gi + (int)b.gx * gj;
    }
    return t;
}

template <class S, int NF, class R> struct TileRegs {
    R v[NF][S::PER];
};

template <class S, int NF, class R>
__device__ __forceinline__ void tile_fetch(TileRegs<S, NF, R> &r, const R *const *src, const TileIdx<S> &t,
                                           long kofs)
{
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const R *plane = src[f] + kofs;
#pragma unroll
        for (int q = 0; q < S::PER; q++) r.v[f][q] = plane[t.off[q]];
    }
}

// LDS layout: [field][slot 0..2][S::N], then a scratch row of S::NT.
template <class S, int NF> constexpr int ring_size() { return NF * 3 * S::N + S::NT; }

template <class S, int NF, class R, class SL>
__device__ __forceinline__ void tile_commit(R *lds, SL slot, const TileRegs<S, NF, R> &r, const TileIdx<S> &t)
{
    (void)t;
#pragma unroll
    for (int f = 0; f < NF; f++)
#pragma unroll
        for (int q = 0; q < S::PER; q++) {
            const int e = threadIdx.x + q * S::NT;
            int li = (f * 3 + (int)slot) * S::N + e;
            if (q == S::PER - 1 && e >= S::N) li = NF * 3 * S::N + (int)threadIdx.x;
            lds[li] = r.v[f][q];
        }
}

template <int V> using IC = std::integral_constant<int, V>;

// ----------------------------------------------------------------- momentum
template <class R, int SRC, int TY, int KB, int UNROLL, int PF = 1, int TX = 64>
struct MomentumMarch {
    static_assert((PF == 1 && (UNROLL == 1 || UNROLL == 3)) || (PF == 2 && UNROLL == 2), "launch shape");
    using S = TileShape<TY, TX>;
    static constexpr int NT = S::NT;

    template <class SM, class SC, class SN>
    __device__ __forceinline__ static void plane(const MomArgs<R> &a, R *lds, TileRegs<S, 4, R> &r,
                                                 const TileIdx<S> &t, const R *const *src, int i, int j, int k,
                                                 int kend, bool active, int c, R (&o)[3], bool xedge, SM sm, SC sc,
                                                 SN sn)
    {
        tile_commit<S, 4>(lds, sn, r, t);   // plane k+1
        __syncthreads();
        if (k + 1 + PF <= kend + 1) tile_fetch<S, 4>(r, src, t, (long)(k + 1 + PF) * a.b.gxy);
        R on[3] = {R(0), R(0), R(0)};
        const long q = active ? a.b.q(i, j, k) : 0;
        const long qs = (long)a.b.nx * a.b.ny;
        if (active && k + 1 <= kend) {
            on[0] = a.dvo0[q + qs];
            on[1] = a.dvo1[q + qs];
            on[2] = a.dvo2[q + qs];
        }
        if (active) {
            auto at = [&](int f) {
                return [=](int di, int dj, int dk) {
                    const int slot = dk < 0 ? (int)sm : (dk > 0 ? (int)sn : (int)sc);
                    return lds[(f * 3 + slot) * S::N + c + dj * S::LX + di];
                };
            };
            auto img = [&](R *f, R v) { march_images(f, a.b, a.img, i, j, k, v, xedge); };
            momentum_cell<1, SRC>(a, i, j, k, at(0), at(1), at(2), at(3), o[0], o[1], o[2], img);
        }
        o[0] = on[0]; o[1] = on[1]; o[2] = on[2];
        __syncthreads();
    }

    __device__ __forceinline__ static void run(const MomArgs<R> &a, R *lds)
    {
        const Box &b = a.b;
        const int bid = xcd_remap(blockIdx.x, gridDim.x);
        const int bx = bid % a.nbx, rest = bid / a.nbx;
        const int by = rest % a.nby, bz = rest / a.nby;
        // a wave is one j row: ty is wave-uniform, so j-dependent branches are scalar
        const int tx = threadIdx.x % S::TX, ty = __builtin_amdgcn_readfirstlane(threadIdx.x / S::TX);
        const bool xedge = bx == 0 || bx == a.nbx - 1;
        const int i0 = bx * S::TX + 1, j0 = by * TY + 1, k0 = bz * KB + 1;
        const int kend = min(k0 + KB - 1, b.nz);
        const int i = i0 + tx, j = j0 + ty;
        const bool active = i <= b.nx && j <= b.ny;
        const int c = (ty + 1) * S::LX + tx + 1;
        const R *src[4] = {a.u, a.v, a.w, a.p};
        const TileIdx<S> t = tile_index<S>(b, i0, j0);
        TileRegs<S, 4, R> r;
        tile_fetch<S, 4>(r, src, t, (long)(k0 - 1) * b.gxy);
        tile_commit<S, 4>(lds, IC<0>{}, r, t);
        tile_fetch<S, 4>(r, src, t, (long)k0 * b.gxy);
        tile_commit<S, 4>(lds, IC<1>{}, r, t);
        tile_fetch<S, 4>(r, src, t, (long)(k0 + 1) * b.gxy);
        TileRegs<S, 4, R> r2;
        if constexpr (PF == 2) {
            if (k0 + 2 <= kend + 1) tile_fetch<S, 4>(r2, src, t, (long)(k0 + 2) * b.gxy);
        }
        R o[3] = {R(0), R(0), R(0)};
        if (active) {
            const long q = b.q(i, j, k0);
            o[0] = a.dvo0[q]; o[1] = a.dvo1[q]; o[2] = a.dvo2[q];
        }
        if constexpr (PF == 2) {
            int sm = 0, sc = 1, sn = 2;
            for (int k = k0; k <= kend; k += 2) {
                plane(a, lds, r, t, src, i, j, k, kend, active, c, o, xedge, sm, sc, sn);
                int tmp = sm;
                sm = sc; sc = sn; sn = tmp;
                if (k + 1 <= kend) {
                    plane(a, lds, r2, t, src, i, j, k + 1, kend, active, c, o, xedge, sm, sc, sn);
                    tmp = sm;
                    sm = sc; sc = sn; sn = tmp;
                }
            }
        } else if constexpr (UNROLL == 3) {
            for (int k = k0; k <= kend; k += 3) {
                plane(a, lds, r, t, src, i, j, k, kend, active, c, o, xedge, IC<0>{}, IC<1>{}, IC<2>{});
                if (k + 1 <= kend) plane(a, lds, r, t, src, i, j, k + 1, kend, active, c, o, xedge, IC<1>{}, IC<2>{}, IC<0>{});
                if (k + 2 <= kend) plane(a, lds, r, t, src, i, j, k + 2, kend, active, c, o, xedge, IC<2>{}, IC<0>{}, IC<1>{});
            }
        } else {
            int sm = 0, sc = 1, sn = 2;
            for (int k = k0; k <= kend; k++) {
                plane(a, lds, r, t, src, i, j, k, kend, active, c, o, xedge, sm, sc, sn);
                const int tmp = sm;
                sm = sc; sc = sn; sn = tmp;
            }
        }
    }
};

// OCC: minimum waves per SIMD the register allocation must allow (1: no limit).
template <class R, int SRC, int TY, int KB, int UNROLL, int PF = 1, int OCC = 1, int TX = 64>
__global__ __launch_bounds__(TX * TY, OCC) void momentum_march_kernel(MomArgs<R> a)
{
    __shared__ R lds[ring_size<TileShape<TY, TX>, 4>()];
    MomentumMarch<R, SRC, TY, KB, UNROLL, PF, TX>::run(a, lds);
}

// --------------------------------------------------------------- projection
// Ring fields: phi, u*, v* (u* and v* need the cell below in i and j for the
// checks); w* and p are prefetched one plane ahead, w* one plane below is
// carried in a register.
template <class R, int SHIFT, int TY, int KB, int UNROLL, int PF = 1, int TX = 64>
struct ProjectMarch {
    static_assert((PF == 1 && (UNROLL == 1 || UNROLL == 3)) || (PF == 2 && UNROLL == 2), "launch shape");
    using S = TileShape<TY, TX>;
    static constexpr int NT = S::NT;

    template <class SM, class SC, class SN>
    __device__ __forceinline__ static void plane(const ProjArgs<R> &a, R *lds, TileRegs<S, 3, R> &r,
                                                 const TileIdx<S> &t, const R *const *src, int i, int j, int k,
                                                 int kend, bool active, int c, double s, double &wsm, double &wsc,
                                                 double &pc, double &md, double &mv, double &bad, bool xedge, SM sm,
                                                 SC sc, SN sn)
    {
        tile_commit<S, 3>(lds, sn, r, t);
        __syncthreads();
        if (k + 1 + PF <= kend + 1) tile_fetch<S, 3>(r, src, t, (long)(k + 1 + PF) * a.b.gxy);
        double wnext = 0.0, pnext = 0.0;
        const long g = a.b.g(i, j, k);
        if (active && k + 1 <= kend) {
            wnext = a.ws[g + a.b.gxy];
            pnext = a.p[g + a.b.gxy];
        }
        if (active) {
            auto L = [&](int f, int di, int dj, int dk) -> double {
                const int slot = dk < 0 ? (int)sm : (dk > 0 ? (int)sn : (int)sc);
                return lds[(f * 3 + slot) * S::N + c + dj * S::LX + di];
            };
            auto F = [&](int di, int dj, int dk) {
                if constexpr (SHIFT) return L(0, di, dj, dk) - s;
                else return L(0, di, dj, dk);
            };
            auto img = [&](R *f, R v) { march_images(f, a.b, a.img, i, j, k, v, xedge); };
            project_cell<1>(a, i, j, k, F, L(1, 0, 0, 0), L(2, 0, 0, 0), wsc, pc, L(1, -1, 0, 0), L(2, 0, -1, 0), wsm, md,
                            mv, bad, img);
        }
        wsm = wsc;
        wsc = wnext;
        pc = pnext;
        __syncthreads();
    }

    __device__ __forceinline__ static void run(const ProjArgs<R> &a, R *lds)
    {
        const Box &b = a.b;
        const int bid = xcd_remap(blockIdx.x, gridDim.x);
        const int bx = bid % a.nbx, rest = bid / a.nbx;
        const int by = rest % a.nby, bz = rest / a.nby;
        // a wave is one j row: ty is wave-uniform, so j-dependent branches are scalar
        const int tx = threadIdx.x % S::TX, ty = __builtin_amdgcn_readfirstlane(threadIdx.x / S::TX);
        const bool xedge = bx == 0 || bx == a.nbx - 1;
        const int i0 = bx * S::TX + 1, j0 = by * TY + 1, k0 = bz * KB + 1;
        const int kend = min(k0 + KB - 1, b.nz);
        const int i = i0 + tx, j = j0 + ty;
        const bool active = i <= b.nx && j <= b.ny;
        const int c = (ty + 1) * S::LX + tx + 1;
        const double s = SHIFT ? a.shift[0] : 0.0;
        double md = -HUGE_VAL, mv = 0.0, bad = 0.0;
        const R *src[3] = {a.phi, a.us, a.vs};
        const TileIdx<S> t = tile_index<S>(b, i0, j0);
        TileRegs<S, 3, R> r;
        tile_fetch<S, 3>(r, src, t, (long)(k0 - 1) * b.gxy);
        tile_commit<S, 3>(lds, IC<0>{}, r, t);
        tile_fetch<S, 3>(r, src, t, (long)k0 * b.gxy);
        tile_commit<S, 3>(lds, IC<1>{}, r, t);
        tile_fetch<S, 3>(r, src, t, (long)(k0 + 1) * b.gxy);
        TileRegs<S, 3, R> r2;
        if constexpr (PF == 2) {
            if (k0 + 2 <= kend + 1) tile_fetch<S, 3>(r2, src, t, (long)(k0 + 2) * b.gxy);
        }
        double wsm = 0.0, wsc = 0.0, pc = 0.0;
        if (active) {
            wsm = a.ws[b.g(i, j, k0 - 1)];
            wsc = a.ws[b.g(i, j, k0)];
            pc = a.p[b.g(i, j, k0)];
        }
        if constexpr (PF == 2) {
            int sm = 0, sc = 1, sn = 2;
            for (int k = k0; k <= kend; k += 2) {
                plane(a, lds, r, t, src, i, j, k, kend, active, c, s, wsm, wsc, pc, md, mv, bad, xedge, sm, sc, sn);
                int tmp = sm;
                sm = sc; sc = sn; sn = tmp;
                if (k + 1 <= kend) {
                    plane(a, lds, r2, t, src, i, j, k + 1, kend, active, c, s, wsm, wsc, pc, md, mv, bad, xedge, sm, sc,
                          sn);
                    tmp = sm;
                    sm = sc; sc = sn; sn = tmp;
                }
            }
        } else if constexpr (UNROLL == 3) {
            for (int k = k0; k <= kend; k += 3) {
                plane(a, lds, r, t, src, i, j, k, kend, active, c, s, wsm, wsc, pc, md, mv, bad, xedge, IC<0>{}, IC<1>{},
                      IC<2>{});
                if (k + 1 <= kend)
                    plane(a, lds, r, t, src, i, j, k + 1, kend, active, c, s, wsm, wsc, pc, md, mv, bad, xedge, IC<1>{},
                          IC<2>{}, IC<0>{});
                if (k + 2 <= kend)
                    plane(a, lds, r, t, src, i, j, k + 2, kend, active, c, s, wsm, wsc, pc, md, mv, bad, xedge, IC<2>{},
                          IC<0>{}, IC<1>{});
            }
        } else {
            int sm = 0, sc = 1, sn = 2;
            for (int k = k0; k <= kend; k++) {
                plane(a, lds, r, t, src, i, j, k, kend, active, c, s, wsm, wsc, pc, md, mv, bad, xedge, sm, sc, sn);
                const int tmp = sm;
                sm = sc; sc = sn; sn = tmp;
            }
        }
        block_max3<NT>(md, mv, bad, a.part, bid);
    }
};

template <class R, int SHIFT, int TY, int KB, int UNROLL, int PF = 1, int OCC = 1, int TX = 64>
__global__ __launch_bounds__(TX * TY, OCC) void project_march_kernel(ProjArgs<R> a)
{
    __shared__ R lds[ring_size<TileShape<TY, TX>, 3>()];
    ProjectMarch<R, SHIFT, TY, KB, UNROLL, PF, TX>::run(a, lds);
}

// The checks of a pending step: project_cell without its stores, on columns of
// cells two rows wide that a thread walks in k, reading x and y neighbours from
// the caches (no LDS, no barrier) and carrying what plane k needs of k - 1; the
// loads of plane k + 2 are in flight while plane k is computed.  HBM bounds it,
// 4 words per cell (the projection's march without its stores -> this: 256^3
// 158 -> 145 us, 128^3 22 -> 18.4).
template <class R, int SHIFT> __global__ __launch_bounds__(256) void project_checks_kernel(ProjArgs<R> a, int kb)
{
    constexpr int TX = 64, TY = 4, NJ = 2;
    const Box &b = a.b;
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int bx = bid % a.nbx, rest = bid / a.nbx, by = rest % a.nby, bz = rest / a.nby;
    const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
    const int i = bx * TX + tx + 1, j = (by * TY + ty) * NJ + 1, k0 = bz * kb + 1, kend = min(k0 + kb - 1, b.nz);
    const double s = SHIFT ? a.shift[0] : 0.0;
    int off[NJ + 2];   // rows j - 1 .. j + NJ; past the grid clamped to its last (values no active cell uses)
#pragma unroll
    for (int r = 0; r < NJ + 2; r++) off[r] = min(i, b.nx) + (int)b.gx * min(j - 1 + r, b.ny + 1);
    struct Plane {
        R f[NJ + 2], fe[NJ], fw[NJ], u[NJ], uw[NJ], v[NJ + 1], w[NJ];
    };
    // plane k; of the one after the march's last only phi is read
    auto load = [&](Plane &p, int k) {
        const long base = (long)k * b.gxy;
        const R *f = a.phi + base, *u = a.us + base, *v = a.vs + base, *w = a.ws + base;
#pragma unroll
        for (int r = 0; r < NJ + 2; r++) p.f[r] = f[off[r]];
        if (k > kend) return;
#pragma unroll
        for (int r = 0; r < NJ + 1; r++) p.v[r] = v[off[r]];
#pragma unroll
        for (int y = 0; y < NJ; y++) {
            p.fe[y] = f[off[y + 1] + 1];
            p.fw[y] = f[off[y + 1] - 1];
            p.u[y] = u[off[y + 1]];
            p.uw[y] = u[off[y + 1] - 1];
            p.w[y] = w[off[y + 1]];
        }
    };
    R fb[NJ], wb[NJ];   // phi and w* of plane k - 1
#pragma unroll
    for (int y = 0; y < NJ; y++) {
        fb[y] = a.phi[off[y + 1] + (long)(k0 - 1) * b.gxy];
        wb[y] = a.ws[off[y + 1] + (long)(k0 - 1) * b.gxy];
    }
    Plane c, n{}, x{};
    load(c, k0);
    load(n, k0 + 1);
    double md = -HUGE_VAL, mv = 0.0, bad = 0.0;
    for (int k = k0; k <= kend; k++) {
        if (k < kend) load(x, k + 2);
#pragma unroll
        for (int y = 0; y < NJ; y++) {
            if (i <= b.nx && j + y <= b.ny) {
                auto F = [&](int di, int dj, int dk) {
                    const R f = di > 0 ? c.fe[y] : di < 0 ? c.fw[y] : dk > 0 ? n.f[y + 1] : dk < 0 ? fb[y] : c.f[y + 1 + dj];
                    if constexpr (SHIFT) return (double)f - s;
                    else return (double)f;
                };
                auto none = [](R *, R) {};
                project_cell<1, R, decltype(F), decltype(none), 0>(a, i, j + y, k, F, c.u[y], c.v[y + 1], c.w[y], 0.0,
                                                                   c.uw[y], c.v[y], wb[y], md, mv, bad, none);
            }
            fb[y] = c.f[y + 1];
            wb[y] = c.w[y];
        }
        c = n;
        n = x;
    }
    block_max3<256>(md, mv, bad, a.part, bid);
}

// ------------------------------------------------- projection + momentum
// Step n's projection and pressure update fused with step n+1's momentum,
// for a grid periodic in every direction.  The state (u, v, w, p) after
// step n is formed tile by tile from u*, v*, w*, p and phi of step n with
// the projection's arithmetic (each value rounded once to R), placed in the
// momentum's 4-field LDS ring and advanced to u*, v*, w* of step n+1; only
// p of step n and the momentum's outputs are stored.  Step n's checks are
// not formed: step n+1 ends pending, and its checks are the ones a reader
// asks for.  Every
// ghost position of the state is the periodic image of an interior cell, so
// tile cells outside the interior are formed at the wrapped interior index:
// the same values the unfused projection writes and its images copy.
// u*, v*, w* and p are read at the cell, phi at the cell and one cell above
// along each axis (phi's face ghosts are its periodic images).
// ZW: the z faces are no-slip walls instead (channel: x, y periodic).  The
// state's ghost planes k = 0 and nz+1 then follow the ghost fill's z rules
// applied to the projected first and last planes: u, v = 2 bc - f (the bc
// planes are indexed at the cell's own, unwrapped (i, j)), w = bc (and the
// last interior w is overwritten with bc), p = the neighbouring interior
// value; a pending mean shift of phi is subtracted as the projection does.
//
// What bounds it: HBM on large grids (256^3 FP64 2.013 GB in 420 us, 4.8
// TB/s, what a device copy reaches and 0.84 of a large FP64 add; 430 to 440 us
// inside a run, the figures here are of launches back to back); on small ones the chain of one plane
// (load, form, barrier, stencil: 2.4 us alone on a CU).  Both ask for more
// work per plane and barrier, so a thread owns two rows: the tile's halo is
// 1.27 instead of 1.52 of its cells, the rows share their neighbours, edge
// products and the face between them, and what plane k needs of k - 1 (the
// thread's own u, v, w and three fluxes) is carried in registers, so the ring
// is read at planes k and k + 1 only and one barrier per plane suffices.
// One row per thread and two barriers took 479 us at 256^3 (FP32 259, now
// 235), 62 at 128^3 (now 49), 43 at 32^3 (now 7); 64 x 16 tiles with four rows
// per thread 453; 64 x 8 with two, 470.
// Loads and stores take a uniform base and a 32-bit offset per element: with
// 64-bit pointers the compiler hoisted some 70 registers of addresses out of
// the march (254 registers, one wave per SIMD; now 209).
template <class R> struct PMArgs {
    MomArgs<R> m;                  // momentum of step n+1 (m.u, m.v, m.w, m.p unused)
    const R *__restrict__ us;      // u*, v*, w* of step n
    const R *__restrict__ vs;
    const R *__restrict__ ws;
    const R *__restrict__ phi;
    const R *__restrict__ p_in;    // p before step n
    R *__restrict__ p_out;         // p after step n (interior)
    const double *shift;           // pending mean of phi (ZW), or null
    const R *zlo[3], *zhi[3];      // ZW: bc planes of u, v, w at the front and back faces
    double pid, pdt, prhof, pirhof;
    int prpow2;
    int kb;                        // planes marched per workgroup
    // ZW == 2 (general walls): non-periodic axes (bit 0 x, 1 y, 2 z); per
    // state field u, v, w, p the bc type of face f in bits 2f..2f+1 and the
    // location (0 centre, 1 x, 2 y, 3 z face) in bits 12..13; and the bc
    // value planes, 6 per field in that order, in device memory
    int wall;
    int gtype[4];
    const R *const *gplane;
    R *wbuf;   // ZW == 2: the state at the wall positions (pm_wall_layout)
    R *save[3];   // SAVE: u, v, w of step n (ghosted, with periodic images)
};

// The general-wall form (ZW == 2).  Along one wall axis a ghosted position
// is the low ghost (0), the high ghost (n + 1) or the high face's
// overwritten normal (n, f(N) = bc): pm_wall_pos gives 0, 1, 2 for these
// and -1 elsewhere.
__device__ __forceinline__ int pm_wall_pos(int g, int n)
{
    return g == 0 ? 0 : (g == n + 1 ? 1 : (g == n ? 2 : -1));
}

// The state at every wall position is formed before the march by
// wall_state_kernel into a face buffer, one block per field of
// pm_wall_layout().per_field values: x section [nz+2][ny+2][3] (kk, gj,
// position px fastest: px = 1 and 2 read the same source cell, so a wave
// reads each of its lines once), y section [3][nz+2][nx+2] (py, kk, gi),
// z section [3][ny+2][nx+2] (pz, gj, gi).  Positions on several walls
// (edges, corners) hold the same value in each section that has them.
struct PMWallLayout {
    long xs, ys, zs;   // section offsets
    long xp, yp, zp;   // words per position plane
    long per_field;
};
__host__ __device__ __forceinline__ PMWallLayout pm_wall_layout(const Box &b)
{
    PMWallLayout w;
    w.xp = (long)(b.ny + 2) * (b.nz + 2);
    w.yp = (long)(b.nx + 2) * (b.nz + 2);
    w.zp = (long)(b.nx + 2) * (b.ny + 2);
    w.xs = 0;
    w.ys = 3 * w.xp;
    w.zs = w.ys + 3 * w.yp;
    w.per_field = w.zs + 3 * w.zp;
    return w;
}

// The ghost value of one state field at ghosted position (gi, gj, kk),
// given v = the field's projected value at the interior cell the ghost fill
// reads, (ix, jy, kz) per axis: the ghost kernel's x -> y -> z composition
// (S1, S2, S3) applied to that value, each level with the value plane
// indexed at that level's coordinates, and the high-face normal overwrite
// f(N) = bc.  Periodic axes only move the index.  gt: packed types and
// location (PMArgs::gtype), pl: the field's 6 planes.
template <class R>
__device__ __forceinline__ R pm_ghost_chain(int gt, const R *const *pl, const Box &b, int wall, int gi, int gj,
                                            int kk, int jy, int kz, R v)
{
    const R two = R(2.0);
    const int loc = (gt >> 12) & 3;   // 1 x, 2 y, 3 z, 0 centre
    auto ty = [&](int f) { return (gt >> (2 * f)) & 3; };
    if (wall & 1) {   // S1(gi, jy, kz)
        const long pj = jy + (long)(b.ny + 2) * kz;
        if (gi == 0) {
            if (ty(0) == 1) v = loc == 1 ? pl[0][pj] : two * pl[0][pj] - v;
        } else if (gi == b.nx + 1) {
            if (ty(1) == 1) v = loc == 1 ? pl[1][pj] : two * pl[1][pj] - v;
        } else if (gi == b.nx && ty(1) == 1 && loc == 1) {
            v = pl[1][pj];
        }
    }
    if (wall & 2) {   // S2(gi, gj, kz)
        const long pi = gi + (long)(b.nx + 2) * kz;
        if (gj == 0) {
            if (ty(2) == 1) v = loc == 2 ? pl[2][pi] : two * pl[2][pi] - v;
        } else if (gj == b.ny + 1) {
            if (ty(3) == 1) v = loc == 2 ? pl[3][pi] : two * pl[3][pi] - v;
        } else if (gj == b.ny && ty(3) == 1 && loc == 2) {
            v = pl[3][pi];
        }
    }
    if (wall & 4) {   // S3(gi, gj, kk)
        const long pij = gi + (long)(b.nx + 2) * gj;
        if (kk == 0) {
            if (ty(4) == 1) v = loc == 3 ? pl[4][pij] : two * pl[4][pij] - v;
        } else if (kk == b.nz + 1) {
            if (ty(5) == 1) v = loc == 3 ? pl[5][pij] : two * pl[5][pij] - v;
        } else if (kk == b.nz && ty(5) == 1 && loc == 3) {
            v = pl[5][pij];
        }
    }
    return v;
}

// Source index of a ghosted coordinate along one axis: periodic wraps,
// a wall axis reads the adjacent interior cell.
__device__ __forceinline__ int pm_src(int g, int n, bool wall)
{
    if (g == 0) return wall ? 1 : n;
    if (g == n + 1) return wall ? n : 1;
    return g;
}

// SAVE (periodic grids): also store u, v, w of step n and their periodic
// images into a.save, for callers that keep every state (the adjoint's
// recomputed segments).
// P2: rhof is a power of two (1/rhof exact), else every division is an IEEE
// divide.  A template parameter: as a run-time test each of the 39 divisions
// of the unrolled body kept its branch and its inlined divide, which split the
// body into some 60 blocks.
template <class R, int SRC, int TY, int ZW, int TX = 64, int SAVE = 0, int NJ = 2, int P2 = 1>
struct ProjectMomentumMarch {
    using S = TileShape<TY, TX, NJ>;
    static constexpr int NT = S::NT, NRAW = 8;
    struct Raw {
        R v[NRAW][S::PER];
        int wl;   // ZW == 2: bit q set when element q took its state from the face buffer
    };
    // ZW == 2: per tile element, its face buffer offset at plane 0 and the
    // stride per plane when it sits on an x or y wall position (ofs < 0
    // otherwise), and its offset in a z position plane
    struct WallIdx {
        int ofs[S::PER], str[S::PER], zo[S::PER];
    };
    struct PlaneIdx {   // ZW: bc plane index i + (nx+2) j of each tile element
        int v[S::PER];
    };

    __device__ __forceinline__ static PlaneIdx plane_index(const Box &b, int i0, int j0)
    {
        PlaneIdx pi{};
        if constexpr (ZW == 1) {
#pragma unroll
            for (int q = 0; q < S::PER; q++) {
                const int e = threadIdx.x + q * S::NT;
                const int ri = e % S::LX, rj = e / S::LX;
                int gi = min(i0 - 1 + ri, b.nx + 1), gj = min(j0 - 1 + rj, b.ny + 1);
                if (e >= S::N) { gi = i0; gj = j0; }
                pi.v[q] = gi + (b.nx + 2) * gj;
            }
        }
        return pi;
    }

    // Tile element offsets at k = 0 with every ghost index wrapped to its
    // periodic interior image (elements past the grid are clamped first).
    __device__ __forceinline__ static TileIdx<S> index(const Box &b, int i0, int j0, int wall)
    {
        TileIdx<S> t;
#pragma unroll
        for (int q = 0; q < S::PER; q++) {
            const int e = threadIdx.x + q * S::NT;
            const int ri = e % S::LX, rj = e / S::LX;
            int gi = min(i0 - 1 + ri, b.nx + 1), gj = min(j0 - 1 + rj, b.ny + 1);
            if (e >= S::N) { gi = i0; gj = j0; }
            if constexpr (ZW == 2) {
                gi = pm_src(gi, b.nx, wall & 1);
                gj = pm_src(gj, b.ny, wall & 2);
            } else {
                gi = gi == 0 ? b.nx : (gi == b.nx + 1 ? 1 : gi);
                gj = gj == 0 ? b.ny : (gj == b.ny + 1 ? 1 : gj);
            }
            t.off[q] = gi + (int)b.gx * gj;
        }
        return t;
    }

    // base[element offset], the offset kept as 32-bit bytes and the base
    // uniform: one address VGPR per element instead of a 64-bit pair per load.
    __device__ __forceinline__ static R at_off(const R *base, unsigned bytes)
    {
        return *reinterpret_cast<const R *>(reinterpret_cast<const char *>(base) + bytes);
    }
    __device__ __forceinline__ static R *to_off(R *base, unsigned bytes)
    {
        return reinterpret_cast<R *>(reinterpret_cast<char *>(base) + bytes);
    }

    __device__ __forceinline__ static void fetch(Raw &r, const PMArgs<R> &a, const TileIdx<S> &t,
                                                 const WallIdx &wi, int kk)
    {
        const Box &b = a.m.b;
        // the interior plane the state at plane kk is formed from
        const int kw = ZW == 1   ? (kk == 0 ? 1 : (kk == b.nz + 1 ? b.nz : kk))
                       : ZW == 2 ? pm_src(kk, b.nz, a.wall & 4)
                                 : (kk == 0 ? b.nz : (kk == b.nz + 1 ? 1 : kk));
        const long kofs = (long)kw * b.gxy;
        const R *bu = a.us + kofs, *bv = a.vs + kofs, *bw = a.ws + kofs, *bp = a.p_in + kofs;
        const R *f0 = a.phi + kofs, *fy = f0 + b.gx, *fz = f0 + b.gxy;
        // ZW == 2: elements on a wall position load u, v, w, p of the face
        // buffer instead (a z wall plane: all of them)
        [[maybe_unused]] int pz = -1;
        [[maybe_unused]] PMWallLayout L{};
        if constexpr (ZW == 2) {
            pz = (a.wall & 4) ? pm_wall_pos(kk, b.nz) : -1;
            L = pm_wall_layout(b);
            r.wl = 0;
        }
#pragma unroll
        for (int q = 0; q < S::PER; q++) {
            const unsigned o = (unsigned)t.off[q] * (unsigned)sizeof(R);
            if constexpr (ZW == 2) {
                const R *su = to_off(const_cast<R *>(bu), o), *sv = to_off(const_cast<R *>(bv), o),
                        *sw = to_off(const_cast<R *>(bw), o), *sp = to_off(const_cast<R *>(bp), o);
                const bool wl = pz >= 0 || wi.ofs[q] >= 0;
                const long ow = pz >= 0 ? L.zs + pz * L.zp + wi.zo[q] : wi.ofs[q] + (long)wi.str[q] * kk;
                if (wl) {
                    const R *w0 = a.wbuf + ow;
                    su = w0; sv = w0 + L.per_field; sw = w0 + 2 * L.per_field; sp = w0 + 3 * L.per_field;
                    r.wl |= 1 << q;
                }
                r.v[0][q] = *su;
                r.v[1][q] = *sv;
                r.v[2][q] = *sw;
                r.v[3][q] = *sp;
            } else {
                r.v[0][q] = at_off(bu, o);
                r.v[1][q] = at_off(bv, o);
                r.v[2][q] = at_off(bw, o);
                r.v[3][q] = at_off(bp, o);
            }
            r.v[4][q] = at_off(f0, o);
            r.v[5][q] = at_off(f0 + 1, o);
            r.v[6][q] = at_off(fy, o);
            r.v[7][q] = at_off(fz, o);
        }
    }

    // The state at tile plane kk (project_cell's arithmetic, then the z wall
    // rules when ZW) into ring slot `slot`.
    template <class SL>
    __device__ __forceinline__ static void commit(R *lds, SL slot, const Raw &r, const PMArgs<R> &a,
                                                  const PlaneIdx &pi, int kk, double sh)
    {
        auto dr = [&](double x) { return over_rho(x, a.prhof, a.pirhof, P2); };
        const int nz = a.m.b.nz;
#pragma unroll
        for (int q = 0; q < S::PER; q++) {
            const int e = threadIdx.x + q * S::NT;
            double f0 = (double)r.v[4][q], fx = (double)r.v[5][q], fy = (double)r.v[6][q], fz = (double)r.v[7][q];
            if constexpr (ZW == 1) {
                f0 = f0 - sh; fx = fx - sh; fy = fy - sh; fz = fz - sh;
            }
            R un = (R)((double)r.v[0][q] - dr((fx - f0) * a.pid * a.pdt));
            R vn = (R)((double)r.v[1][q] - dr((fy - f0) * a.pid * a.pdt));
            R wn = (R)((double)r.v[2][q] - dr((fz - f0) * a.pid * a.pdt));
            R pn = (R)((double)r.v[3][q] + f0);
            if constexpr (ZW == 2) {
                if (r.wl & (1 << q)) {   // the face buffer's final state
                    un = r.v[0][q]; vn = r.v[1][q]; wn = r.v[2][q]; pn = r.v[3][q];
                }
            }
            if constexpr (ZW == 1) {
                const R two = R(2.0);
                if (kk == 0) {
                    un = two * a.zlo[0][pi.v[q]] - un;
                    vn = two * a.zlo[1][pi.v[q]] - vn;
                    wn = a.zlo[2][pi.v[q]];
                } else if (kk >= nz) {
                    if (kk > nz) {
                        un = two * a.zhi[0][pi.v[q]] - un;
                        vn = two * a.zhi[1][pi.v[q]] - vn;
                    }
                    wn = a.zhi[2][pi.v[q]];
                }
            }
            const R vals[4] = {un, vn, wn, pn};
#pragma unroll
            for (int f = 0; f < 4; f++) {
                int li = (f * 3 + (int)slot) * S::N + e;
                if (q == S::PER - 1 && e >= S::N) li = 4 * 3 * S::N + (int)threadIdx.x;
                lds[li] = vals[f];
            }
        }
    }

    // ZW == 2: the face buffer offsets of this thread's tile elements.
    __device__ __forceinline__ static WallIdx wall_index(const PMArgs<R> &a, int i0, int j0)
    {
        WallIdx wi{};
        if constexpr (ZW == 2) {
            const Box &b = a.m.b;
            const PMWallLayout L = pm_wall_layout(b);
#pragma unroll
            for (int q = 0; q < S::PER; q++) {
                const int e = threadIdx.x + q * S::NT;
                const int ri = e % S::LX, rj = e / S::LX;
                int gi = min(i0 - 1 + ri, b.nx + 1), gj = min(j0 - 1 + rj, b.ny + 1);
                if (e >= S::N) { gi = i0; gj = j0; }
                const int px = (a.wall & 1) ? pm_wall_pos(gi, b.nx) : -1;
                const int py = (a.wall & 2) ? pm_wall_pos(gj, b.ny) : -1;
                wi.zo[q] = gi + (b.nx + 2) * gj;
                if (px >= 0) {
                    wi.ofs[q] = (int)(L.xs + px + 3 * gj);
                    wi.str[q] = 3 * (b.ny + 2);
                } else if (py >= 0) {
                    wi.ofs[q] = (int)(L.ys + py * L.yp + gi);
                    wi.str[q] = b.nx + 2;
                } else {
                    wi.ofs[q] = -1;
                    wi.str[q] = 0;
                }
            }
        }
        return wi;
    }

    // What the march carries from plane k - 1 to plane k in registers: the
    // thread's own u, v, w at k - 1 and the three fluxes through its cells'
    // k - 1/2 faces (the k + 1/2 fluxes of the plane before, bit for bit).
    struct Carry {
        R um[NJ], vm[NJ], wm[NJ];
        R fu[NJ], fv[NJ], fw[NJ];
    };

    // The carry into plane k from slots sm (plane k - 1) and sc (plane k).
    __device__ __forceinline__ static void start(const R *lds, int sm, int sc, int c, Carry &x)
    {
        const R c025 = R(0.25);
        auto at = [&](int f, int slot, int di, int dj) { return lds[(f * 3 + slot) * S::N + c + dj * S::LX + di]; };
#pragma unroll
        for (int r = 0; r < NJ; r++) {
            const R um = at(0, sm, 0, r), vm = at(1, sm, 0, r), wm = at(2, sm, 0, r), wc = at(2, sc, 0, r);
            x.um[r] = um; x.vm[r] = vm; x.wm[r] = wm;
            x.fu[r] = ((at(0, sc, 0, r) + um) * (at(2, sm, 1, r) + wm)) * c025;
            x.fv[r] = ((at(1, sc, 0, r) + vm) * (at(2, sm, 0, r + 1) + wm)) * c025;
            x.fw[r] = ((wm + wc) * (wm + wc)) * c025;
        }
    }

    // march_images() from a uniform base: v to every periodic image (axes
    // `ax`) of cell (i, j, k), whose row starts at `row` (uniform) and whose
    // in-plane byte offset is gb; xb is the offset of its x image.  Only
    // uniform values are hoisted out of the march (64-bit image addresses
    // per lane would be, and would live through it).
    __device__ __forceinline__ static void images(R *row, const Box &b, int ax, int j, int k, unsigned gb, unsigned xb,
                                                  bool xi, R v)
    {
        if ((ax & 1) && xi) *to_off(row, xb) = v;
        const bool yj = (ax & 2) && (j == 1 || j == b.ny);
        const bool zk = (ax & 4) && (k == 1 || k == b.nz);
        if (yj || zk) {
            const long dy = (j == 1 ? b.ny : -b.ny) * b.gx, dz = (k == 1 ? b.nz : -b.nz) * b.gxy;
            auto put = [&](R *to) {
                *to_off(to, gb) = v;
                if ((ax & 1) && xi) *to_off(to, xb) = v;
            };
            if (yj) put(row + dy);
            if (zk) put(row + dz);
            if (yj && zk) put(row + dy + dz);
        }
    }

    // Momentum of the thread's NJ cells at plane k (slots sc: k, sn: k + 1).
    // momentum_cell's expressions; each flux two of the cells or two of the
    // equations share (u v on the z edges: u's y flux and v's x flux; u w; v
    // w; a face between the thread's rows) is formed once.
    __device__ __forceinline__ static void momentum(const PMArgs<R> &a, const R *lds, int sc, int sn, int c, int i,
                                                    int j, int k, bool active, bool xedge, Carry &x,
                                                    const R (&o)[3][NJ])
    {
        const MomArgs<R> &m = a.m;
        const R id = m.id, id2 = m.id2, c0 = R(0.0), c025 = R(0.25), c2 = R(2.0);
        const R A = m.A, B = m.B, dt = m.dt;
        auto at = [&](int f, int slot, int di, int dj) { return lds[(f * 3 + slot) * S::N + c + dj * S::LX + di]; };
        auto dr = [&](R v) { return over_rho(v, m.rhof, m.irhof, P2); };
        // in-plane byte offsets of cell (i, j); planes and rows move the uniform base
        const unsigned gb = (unsigned)((i + (int)m.b.gx * j) * (int)sizeof(R));
        const unsigned qb = (unsigned)(((i - 1) + m.b.nx * (j - 1)) * (int)sizeof(R));
        const bool xi = xedge && (i == 1 || i == m.b.nx);
        const unsigned xb = i == 1 ? gb + (unsigned)(m.b.nx * (int)sizeof(R)) : gb - (unsigned)(m.b.nx * (int)sizeof(R));
        const long gk = (long)k * m.b.gxy, qk = (long)(k - 1) * m.b.nx * m.b.ny;
        R U[NJ + 2], V[NJ + 2], W[NJ + 2], V1[NJ + 1], Ul[NJ + 1], P[NJ + 1];   // rows -1 .. NJ at [row + 1]
#pragma unroll
        for (int r = -1; r <= NJ; r++) {
            U[r + 1] = at(0, sc, 0, r);
            V[r + 1] = at(1, sc, 0, r);
            W[r + 1] = at(2, sc, 0, r);
        }
#pragma unroll
        for (int r = 0; r <= NJ; r++) {
            V1[r] = at(1, sc, 1, r - 1);   // v at i + 1, rows -1 .. NJ - 1
            Ul[r] = at(0, sc, -1, r);      // u at i - 1, rows 0 .. NJ
            P[r] = at(3, sc, 0, r);
        }
        R exy[NJ + 1], fyy[NJ + 1];   // u v on the edge and v v through the face above rows -1 .. NJ - 1
#pragma unroll
        for (int r = 0; r <= NJ; r++) {
            const R vv = V[r + 1] + V[r];
            exy[r] = ((U[r + 1] + U[r]) * (V1[r] + V[r])) * c025;
            fyy[r] = c025 * (vv * vv);
        }
        R vwlo = ((W[1] + W[0]) * (V[0] + at(1, sn, 0, -1))) * c025;   // v w on the edge below row 0
#pragma unroll
        for (int r = 0; r < NJ; r++) {
            const R u0 = U[r + 1], v0 = V[r + 1], w0 = W[r + 1];
            const R ur = at(0, sc, 1, r), ul = Ul[r], un = at(0, sn, 0, r), vn = at(1, sn, 0, r), wn = at(2, sn, 0, r);
            const R wr = at(2, sc, 1, r), wl = at(2, sc, -1, r);
            const R uwkp = ((un + u0) * (wr + w0)) * c025;
            const R vwkp = ((vn + v0) * (W[r + 2] + w0)) * c025;
            const R wwkp = ((w0 + wn) * (w0 + wn)) * c025;
            const long g = gk + r * m.b.gx, q = qk + (long)r * m.b.nx;   // + the cell's in-plane offset
            const bool live = active && j + r <= m.b.ny;
            auto put = [&](R *us, R *dvo, R val, R dv) {
                if (live) {
                    *to_off(us + g, gb) = val;
                    images(us + g, m.b, m.img, j + r, k, gb, xb, xi, val);
                    store_stream(to_off(dvo + q, qb), dv);
                }
            };
            // ---- x momentum
            {
                const R uuip = c025 * ((ur + u0) * (ur + u0)), uuim = c025 * ((ul + u0) * (ul + u0));
                R s = (c0 - (uuip - uuim) * id) - (exy[r + 1] - exy[r]) * id;
                s = s - (uwkp - x.fu[r]) * id;
                R l = (((ur - c2 * u0) + ul) + ((U[r + 2] - c2 * u0) + U[r])) * id2;
                l = l + ((un - c2 * u0) + x.um[r]) * id2;
                s = s + dr(m.mu * l);
                if constexpr (SRC) s = s + dr(live ? at_off(m.s0 + q, qb) : c0);
                else s = s + c0;
                const R gp = (at(3, sc, 1, r) - P[r]) * id;
                const R rhs = ((-dr(gp) + A * s) + B * o[0][r]) + m.g0;
                put(m.us, m.dvo0, u0 + dt * rhs, s);
            }
            // ---- y momentum
            {
                const R vl = at(1, sc, -1, r);
                const R vuim = ((v0 + vl) * (Ul[r + 1] + ul)) * c025;
                R s = (c0 - (exy[r + 1] - vuim) * id) - (fyy[r + 1] - fyy[r]) * id;
                s = s - (vwkp - x.fv[r]) * id;
                R l = (((V1[r + 1] - c2 * v0) + vl) + ((V[r + 2] - c2 * v0) + V[r])) * id2;
                l = l + ((vn - c2 * v0) + x.vm[r]) * id2;
                s = s + dr(m.mu * l);
                if constexpr (SRC) s = s + dr(live ? at_off(m.s1 + q, qb) : c0);
                else s = s + c0;
                const R gp = (P[r + 1] - P[r]) * id;
                const R rhs = ((-dr(gp) + A * s) + B * o[1][r]) + m.g1;
                put(m.vs, m.dvo1, v0 + dt * rhs, s);
            }
            // ---- z momentum
            {
                const R wuim = ((w0 + wl) * (ul + at(0, sn, -1, r))) * c025;
                R s = ((c0 - (uwkp - wuim) * id) - (vwkp - vwlo) * id) - (wwkp - x.fw[r]) * id;
                const R l = ((((wr - c2 * w0) + wl) + ((W[r + 2] - c2 * w0) + W[r])) + ((wn - c2 * w0) + x.wm[r])) * id2;
                s = s + dr(m.mu * l);
                if constexpr (SRC) s = s + dr(live ? at_off(m.s2 + q, qb) : c0);
                else s = s + c0;
                const R gp = (at(3, sn, 0, r) - P[r]) * id;
                const R rhs = ((-dr(gp) + A * s) + B * o[2][r]) + m.g2;
                put(m.ws, m.dvo2, w0 + dt * rhs, s);
            }
            if (live) store_stream(to_off(a.p_out + g, gb), P[r]);
            if constexpr (SAVE) {
                if (live) {
                    const R st[3] = {u0, v0, w0};
#pragma unroll
                    for (int f = 0; f < 3; f++) {
                        *to_off(a.save[f] + g, gb) = st[f];
                        images(a.save[f] + g, m.b, 7, j + r, k, gb, xb, xi, st[f]);
                    }
                }
            }
            vwlo = vwkp;
            x.um[r] = u0; x.vm[r] = v0; x.wm[r] = w0;
            x.fu[r] = uwkp; x.fv[r] = vwkp; x.fw[r] = wwkp;
        }
    }

    __device__ __forceinline__ static void run(const PMArgs<R> &a, R *lds)
    {
        const MomArgs<R> &m = a.m;
        const Box &b = m.b;
        const int bid = xcd_remap(blockIdx.x, gridDim.x);
        const int bx = bid % m.nbx, rest = bid / m.nbx;
        const int by = rest % m.nby, bz = rest / m.nby;
        const int tx = threadIdx.x % S::TX, ty = __builtin_amdgcn_readfirstlane(threadIdx.x / S::TX);
        const bool xedge = bx == 0 || bx == m.nbx - 1;
        const int i0 = bx * S::TX + 1, j0 = by * TY + 1, k0 = bz * a.kb + 1;
        const int kend = min(k0 + a.kb - 1, b.nz);
        const int i = i0 + tx, j = j0 + NJ * ty;
        const bool active = i <= b.nx && j <= b.ny;
        const int c = (NJ * ty + 1) * S::LX + tx + 1;
        const TileIdx<S> t = index(b, i0, j0, a.wall);
        const PlaneIdx pi = plane_index(b, i0, j0);
        const double sh = (ZW == 1 && a.shift) ? a.shift[0] : 0.0;
        const long qs = (long)b.nx * b.ny;
        Raw r;
        const WallIdx wi = wall_index(a, i0, j0);
        fetch(r, a, t, wi, k0 - 1);
        commit(lds, 0, r, a, pi, k0 - 1, sh);
        fetch(r, a, t, wi, k0);
        commit(lds, 1, r, a, pi, k0, sh);
        fetch(r, a, t, wi, k0 + 1);
        // dv_o of the thread's cells at plane k (a cell past the grid reads the plane's first)
        unsigned ob[NJ];
#pragma unroll
        for (int y = 0; y < NJ; y++)
            ob[y] = active && j + y <= b.ny ? (unsigned)(((i - 1) + b.nx * (j + y - 1)) * (int)sizeof(R)) : 0u;
        auto old = [&](R (&o)[3][NJ], int k) {
            const long qk = (long)(k - 1) * qs;
#pragma unroll
            for (int y = 0; y < NJ; y++) {
                o[0][y] = load_stream(to_off(m.dvo0 + qk, ob[y]));
                o[1][y] = load_stream(to_off(m.dvo1 + qk, ob[y]));
                o[2][y] = load_stream(to_off(m.dvo2 + qk, ob[y]));
            }
        };
        R o[3][NJ];
        old(o, k0);
        Carry x;
        __syncthreads();
        start(lds, 0, 1, c, x);
        int sm = 0, sc = 1, sn = 2;
        // One barrier per plane: plane k reads slots k and k + 1 (what it needs
        // of k - 1 is carried), so the next plane's commit, into the slot of
        // k - 1, may run beside it; the barrier of plane k stands between that
        // commit and every read of slot k - 1.
        for (int k = k0; k <= kend; k++) {
            commit(lds, sn, r, a, pi, k + 1, sh);   // state at plane k+1
            __syncthreads();
            if (k < kend) fetch(r, a, t, wi, k + 2);
            R on[3][NJ] = {};
            if (k < kend) old(on, k + 1);
            // p of step n; its checks are not formed here: the step ends
            // pending, and a read of the scalars runs the checks-only pass
            momentum(a, lds, sc, sn, c, i, j, k, active, xedge, x, o);
#pragma unroll
            for (int f = 0; f < 3; f++)
#pragma unroll
                for (int y = 0; y < NJ; y++) o[f][y] = on[f][y];
            const int tmp = sm;
            sm = sc; sc = sn; sn = tmp;
        }
    }
};

template <class R, int SRC, int ZW, int TY, int OCC, int TX, int SAVE, int NJ, int P2>
__global__ __launch_bounds__(TX *TY / NJ, OCC) void project_momentum_kernel(PMArgs<R> a)
{
    __shared__ R lds[ring_size<TileShape<TY, TX, NJ>, 4>()];
    ProjectMomentumMarch<R, SRC, TY, ZW, TX, SAVE, NJ, P2>::run(a, lds);
}

// The general-wall form's face buffer: u, v, w, p of step n at every wall
// position (pm_wall_layout), one thread per position and field (blockIdx.y).
// Each is the projection of the interior cell the ghost fill reads (commit()'s
// arithmetic, so interior positions such as the overwritten face n match
// the march's own values bit for bit), then the ghost fill's rule chain.
// Latency bounds it, and the fetch of its code: one field per thread is a
// third of the code of four (128 x 128 x 160 nnn: 11.7 -> 9.6 us; 128 x 256 x
// 101 npn, where the x faces' rows, a line per value, weigh more: 11.5 -> 11.8).
template <class R>
__global__ __launch_bounds__(256) void wall_state_kernel(PMArgs<R> a)
{
    const Box &b = a.m.b;
    const PMWallLayout L = pm_wall_layout(b);
    const unsigned idx = blockIdx.x * 256u + threadIdx.x;
    const int f = blockIdx.y;
    if ((long)idx >= L.per_field) return;
    auto coord = [](int pos, int n) { return pos == 0 ? 0 : (pos == 1 ? n + 1 : n); };
    int gi, gj, kk;
    if ((long)idx < L.ys) {
        if (!(a.wall & 1)) return;
        const unsigned rem = idx / 3u, h = (unsigned)b.ny + 2u;
        kk = (int)(rem / h);
        gj = (int)(rem % h);
        gi = coord((int)(idx % 3u), b.nx);
    } else if ((long)idx < L.zs) {
        if (!(a.wall & 2)) return;
        const unsigned at = idx - (unsigned)L.ys, pos = at / (unsigned)L.yp, rem = at % (unsigned)L.yp;
        const unsigned h = (unsigned)b.nx + 2u;
        kk = (int)(rem / h);
        gi = (int)(rem % h);
        gj = coord((int)pos, b.ny);
    } else {
        if (!(a.wall & 4)) return;
        const unsigned at = idx - (unsigned)L.zs, pos = at / (unsigned)L.zp, rem = at % (unsigned)L.zp;
        const unsigned h = (unsigned)b.nx + 2u;
        gj = (int)(rem / h);
        gi = (int)(rem % h);
        kk = coord((int)pos, b.nz);
    }
    const int ix = pm_src(gi, b.nx, a.wall & 1), jy = pm_src(gj, b.ny, a.wall & 2), kz = pm_src(kk, b.nz, a.wall & 4);
    const long o = ix + (long)b.gx * jy + (long)b.gxy * kz;
    auto dr = [&](double x) { return over_rho(x, a.prhof, a.pirhof, a.prpow2); };
    const R *src = f == 0 ? a.us : (f == 1 ? a.vs : (f == 2 ? a.ws : a.p_in));
    const long up = f == 0 ? 1 : (f == 1 ? b.gx : (f == 2 ? b.gxy : 0));
    const int gt = f == 0 ? a.gtype[0] : (f == 1 ? a.gtype[1] : (f == 2 ? a.gtype[2] : a.gtype[3]));
    const double v0 = (double)src[o], f0 = (double)a.phi[o], fu = (double)a.phi[o + up];
    const R st = f == 3 ? (R)(v0 + f0) : (R)(v0 - dr((fu - f0) * a.pid * a.pdt));
    a.wbuf[f * L.per_field + idx] = pm_ghost_chain(gt, a.gplane + 6 * f, b, a.wall, gi, gj, kk, jy, kz, st);
}

}  // namespace fen
