// tridiag_kernels.hip -- batched tridiagonal solves with each column held in
// the registers of a workgroup (FP64 arithmetic for every storage type).
//
// The columns are constant-coefficient: sub- and superdiagonal a = 1/delta^2,
// diagonal -2a + (mwx + mwy) with its first and last entries set by the
// boundary (reference src/poisson.f90:214-226, 741-757, 1094-1135).  The
// Thomas sweep's two recurrences,
//   d_k = (r_k - a d_{k-1}) f_k,  f_k = 1 / (b_k - a c1_{k-1}),  c1_k = a f_k,
//   x_k = d_k - c1_k x_{k+1},
// (2-D: divided by the pivot) are first-order and linear in the carried value,
// so a column is cut into chunks of M rows, one thread each: every thread runs
// its chunk from a zero carry, keeping only the end value and the product of
// the multipliers; the chunks' (product, end) pairs go through LDS, each thread
// folds those before (behind) its own into its carry, and runs the chunk again
// from it.  The multipliers are at most 1 in magnitude, so the products only
// shrink.
#include <cmath>
#include <stdexcept>

#include "fen_internal.hpp"

namespace fen {

namespace {

__host__ __device__ __forceinline__ double2 t_load(double2 v) { return v; }
__host__ __device__ __forceinline__ double2 t_load(float2 v) { return double2{(double)v.x, (double)v.y}; }
__host__ __device__ __forceinline__ double t_load(double v) { return v; }
__device__ __forceinline__ double2 t_mul(double2 a, double f) { return double2{a.x * f, a.y * f}; }
__device__ __forceinline__ double t_mul(double a, double f) { return a * f; }
__device__ __forceinline__ double2 t_div(double2 a, double f) { return double2{a.x / f, a.y / f}; }
__device__ __forceinline__ double t_div(double a, double f) { return a / f; }
__device__ __forceinline__ double2 t_sub(double2 a, double2 b) { return double2{a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ double t_sub(double a, double b) { return a - b; }
__device__ __forceinline__ double2 t_add(double2 a, double2 b) { return double2{a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ double t_add(double a, double b) { return a + b; }
__device__ __forceinline__ void t_store(double2 *p, double2 v) { *p = v; }
__device__ __forceinline__ void t_store(float2 *p, double2 v) { *p = float2{(float)v.x, (float)v.y}; }
__device__ __forceinline__ void t_store(double *p, double v) { *p = v; }

// Column t = o*ni + q starts at o*os + q and has stride s and length n; its
// diagonal shift is mwx[o] + mwy[q] (2-D: mwx[o]).  c1: in 3-D c1[(c - 1)*ncol
// + t] is the c1 of the row before chunk c; in 2-D c1[t*n + k] is every row's.
struct ChunkArgs {
    void *x;
    const double *c1;
    long ncol, ni, os, s;
    int n, nch;
    const double *mwx, *mwy;
    double a, b0, bi, bn;   // off-diagonal; diagonal of the first, inner and last rows
};

// CW adjacent columns per workgroup, nch chunks of M rows each (CW*nch
// threads, adjacent threads on adjacent columns, so every row of the tile is
// one contiguous run).
//
// What bounds it: HBM.  The column is read once and written once (32 B per
// complex element, 16 per real one); c1 is not read but formed again inside
// the chunk from its start (one division per row, hidden).  One thread per
// column moved 72 B (d written and read back, c1 read) and had a tenth of the
// chip's threads: in a run 512 x 256 x 192 ppn 187 -> 88 us (4.6 TB/s), 128 x
// 128 x 160 nnn 54 -> 17, 128 x 256 x 101 npn 47 -> 17; FP32 512 x 512 x 256,
// whose d went through an FP64 scratch, 458 -> 179.
//
// The workgroup of the singular column (mwx + mwy = 0: column 0) runs its
// chunks one after the other instead, in the sweep's own order: whether the
// last pivot of that column is exactly zero is then the sweep's own, and when
// it is not, so is what round-off leaves (but for the last row's quotient,
// here a product with the reciprocal as on every other row).
//
// D2: the 2-D solvers (pn, nn), a few hundred contiguous columns bound by the
// latency of one sweep: c1 is read (formed once per context, by divisions, so
// the singular column's is exactly -1 and its last pivot exactly 0, and the
// column needs no order of its own), and its rows are divided by their pivots,
// as the 2-D sweep's: all rows of the singular column have the same pivot, and
// the error of one rounded reciprocal would sum up over them (700 rows at a
// spacing that is no power of two: 11 times the round-off).  One wave per
// column with the sweep on one or two of its lanes took 70 us at 512 rows and
// 29 at 200, now 9.2 and 5.9 (with reciprocals 8.5 and 5.6).
template <class E, int M, int CW, int NT, int OCC, int D2>
__global__ __launch_bounds__(NT, OCC) void thomas_chunk_kernel(ChunkArgs p)
{
    using A = decltype(t_load(E{}));
    extern __shared__ double2 lds[];
    A *se = reinterpret_cast<A *>(lds);                          // end value of each chunk
    double *sp = reinterpret_cast<double *>(se + (size_t)CW * p.nch);   // product of its multipliers
    const int col = threadIdx.x % CW, ch = threadIdx.x / CW;
    const long t = (long)blockIdx.x * CW + col;
    const bool live = t < p.ncol;
    const long tt = live ? t : p.ncol - 1;   // a valid column: loads kept, nothing stored
    const long o = tt / p.ni, q = tt - o * p.ni;
    const int k0 = ch * M, n = p.n;
    E *x = static_cast<E *>(p.x) + o * p.os + q + (long)k0 * p.s;
    A r[M];
#pragma unroll
    for (int u = 0; u < M; u++) {
        const A v = t_load(x[(long)(k0 + u < n ? u : 0) * p.s]);
        r[u] = k0 + u < n ? v : A{};
    }
    const double mx = p.mwx[o], my = D2 ? 0.0 : p.mwy[q], a0 = ch > 0 ? p.a : 0.0;
    double f[M], g[D2 ? M : 1];   // 1/pivot; D2: the pivot, and the stored c1
    double cp = 0.0;
    if constexpr (D2) {
        const double *c1 = p.c1 + tt * n;
        if (ch > 0) cp = c1[k0 - 1];
#pragma unroll
        for (int u = 0; u < M; u++) g[u] = k0 + u < n - 1 ? c1[k0 + u] : 0.0;
    } else if (ch > 0) {
        cp = p.c1[(long)(ch - 1) * p.ncol + tt];
    }
    auto row = [](A x, double by) {
        if constexpr (D2) return t_div(x, by);
        else return t_mul(x, by);
    };
    double P = 1.0;
    A e{};
#pragma unroll
    for (int u = 0; u < M; u++) {
        const int k = k0 + u;
        const double b = (u == 0 && k == 0) ? p.b0 : (k == n - 1 ? p.bn : p.bi);
        const double ak = u == 0 ? a0 : p.a;
        const double piv = ((b + mx) + my) - ak * cp;
        // a zero last pivot gives 0; rows past the end too
        if constexpr (D2) {
            f[u] = (k < n && piv != 0.0) ? piv : HUGE_VAL;
            cp = g[u];
            P = -g[u] * P;   // a / pivot (the first row's enters no carry, and the last's)
        } else {
            f[u] = (k < n && piv != 0.0) ? 1.0 / piv : 0.0;
            cp = p.a * f[u];
            P = -(ak * f[u]) * P;
        }
        e = row(t_sub(r[u], t_mul(e, ak)), f[u]);
    }
    auto forward = [&](A d) {
#pragma unroll
        for (int u = 0; u < M; u++) {
            d = row(t_sub(r[u], t_mul(d, u == 0 ? a0 : p.a)), f[u]);
            r[u] = d;
        }
        return d;
    };
    auto c1 = [&](int u) { return D2 ? g[D2 ? u : 0] : (k0 + u < n - 1 ? p.a * f[u] : 0.0); };
    auto backward = [&](A v) {
#pragma unroll
        for (int u = M - 1; u >= 0; u--) {
            v = t_sub(r[u], t_mul(v, c1(u)));
            r[u] = v;
        }
        return v;
    };
    if (!D2 && blockIdx.x == 0) {
        for (int c = 0; c < p.nch; c++) {
            if (ch == c) se[c * CW + col] = forward(c > 0 ? se[(c - 1) * CW + col] : A{});
            __syncthreads();
        }
        for (int c = p.nch - 1; c >= 0; c--) {
            if (ch == c) se[c * CW + col] = backward(c < p.nch - 1 ? se[(c + 1) * CW + col] : A{});
            __syncthreads();
        }
    } else {
        se[ch * CW + col] = e;
        sp[ch * CW + col] = P;
        __syncthreads();
        A v{};
        for (int c = 0; c < ch; c++) v = t_add(se[c * CW + col], t_mul(v, sp[c * CW + col]));
        forward(v);
        P = 1.0;
        e = A{};
#pragma unroll
        for (int u = M - 1; u >= 0; u--) {
            e = t_sub(r[u], t_mul(e, c1(u)));
            P = -c1(u) * P;
        }
        __syncthreads();   // every carry has been read
        se[ch * CW + col] = e;
        sp[ch * CW + col] = P;
        __syncthreads();
        v = A{};
        for (int c = p.nch - 1; c > ch; c--) v = t_add(se[c * CW + col], t_mul(v, sp[c * CW + col]));
        backward(v);
    }
    if (!live) return;
#pragma unroll
    for (int u = 0; u < M; u++)
        if (k0 + u < n) t_store(&x[(long)u * p.s], r[u]);
}

// c1 of the last row of every chunk but the last (thomas_chunk_kernel's c1 in 3-D).
__global__ __launch_bounds__(256) void thomas_starts_kernel(ChunkArgs p, double *c1s, int m)
{
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t >= p.ncol) return;
    const double mx = p.mwx[t / p.ni], my = p.mwy[t % p.ni];
    double cp = 0.0;
    for (int k = 0; k < (p.nch - 1) * m; k++) {
        const double piv = (((k == 0 ? p.b0 : p.bi) + mx) + my) - (k == 0 ? 0.0 : p.a) * cp;
        cp = p.a * (1.0 / piv);
        if ((k + 1) % m == 0) c1s[(long)((k + 1) / m - 1) * p.ncol + t] = cp;
    }
}

// The c1 of every row of the columns, for the 2-D form (divisions, the
// reference's association (b - a c1) + mx, src/poisson.f90:346-360).
__global__ __launch_bounds__(256) void thomas_c1_kernel(ChunkArgs p, double *c1)
{
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t >= p.ncol) return;
    const double mx = p.mwx[t / p.ni];
    c1 += t * p.n;
    double cp = p.a / (p.b0 + mx);
    c1[0] = cp;
    for (int k = 1; k < p.n - 1; k++) {
        cp = p.a / ((p.bi - p.a * cp) + mx);
        c1[k] = cp;
    }
}

// How a solver's columns are cut: M rows per chunk, CW columns per workgroup.
struct ChunkPlan {
    int m, cw, nt;
    bool d2;
};

// Complex columns: chunks of 8 rows, 8 columns (128 B runs): 56 us at 512 x
// 256 x 192 against 71 with 16 columns of 12 rows at 256 rows, where the
// larger workgroups fill a CU less evenly.  Real ones: 16 rows, 16 columns (46
// us at 256^3, 50 with 8 rows, 66 with 8 columns).  Columns of more than 512
// rows take 16-row chunks of 8 columns, so that a workgroup keeps to 512
// threads.
ChunkPlan chunk_plan(int solver, int n)
{
    const bool d2 = solver == FEN_SOLVER_PN || solver == FEN_SOLVER_NN;
    if (d2) return ChunkPlan{8, 1, 512, true};
    if (n > 512) return ChunkPlan{16, 8, 512, false};
    if (solver == FEN_SOLVER_NNN) return ChunkPlan{16, 16, 512, false};
    return ChunkPlan{8, 8, 512, false};
}

ChunkArgs chunk_args(fen_ctx *c, const ChunkPlan &pl)
{
    ChunkArgs a{};
    a.c1 = c->d_c1;
    a.mwx = c->d_mwx;
    a.mwy = c->d_mwy;
    a.a = c->tri_a;
    a.b0 = c->tri_b0;
    a.bi = c->tri_bi;
    a.bn = c->tri_bn;
    const int hy = c->ny / 2 + 1;
    switch (c->solver) {
    case FEN_SOLVER_PN:   // complex [kx][j], columns along j
        a.x = c->d_spec;
        a.ncol = c->hx; a.ni = 1; a.os = c->ny; a.s = 1; a.n = c->ny;
        break;
    case FEN_SOLVER_NN:   // real [kx][j]
        a.x = c->d_spec;
        a.ncol = c->nx; a.ni = 1; a.os = c->ny; a.s = 1; a.n = c->ny;
        break;
    case FEN_SOLVER_NPN:  // complex [k][kx][jy], columns along k: column kx hy + jy, one k row contiguous
        a.x = c->d_spec2;
        a.ncol = (long)c->nx * hy; a.ni = hy; a.os = hy; a.s = (long)c->nx * hy; a.n = c->nz;
        break;
    case FEN_SOLVER_NNN:  // real [k][kx][j]
        a.x = c->d_spec;
        a.ncol = (long)c->nx * c->ny; a.ni = c->ny; a.os = c->ny; a.s = (long)c->nx * c->ny; a.n = c->nz;
        break;
    case FEN_SOLVER_PPN:  // complex [kx][k][j]
        a.x = c->d_spec;
        a.ncol = (long)c->hx * c->ny; a.ni = c->ny; a.os = (long)c->ny * c->nz; a.s = c->ny; a.n = c->nz;
        break;
    default: throw std::runtime_error("not a tridiagonal solver");
    }
    if (a.n < 2) throw std::runtime_error("the tridiagonal direction needs at least 2 cells");
    a.nch = (a.n + pl.m - 1) / pl.m;
    return a;
}

template <class E, int M, int CW, int OCC, int D2> void launch_chunks_n(fen_ctx *c, const ChunkArgs &a)
{
    using A = decltype(t_load(E{}));
    const unsigned wgs = (unsigned)((a.ncol + CW - 1) / CW);
    const size_t lds = (size_t)CW * a.nch * (sizeof(A) + sizeof(double));
    hipLaunchKernelGGL((thomas_chunk_kernel<E, M, CW, 512, OCC, D2>), dim3(wgs), dim3((unsigned)(CW * a.nch)), lds,
                       c->stream, a);
}

}  // namespace

// Rows a column may have for thomas_chunk_kernel; longer ones keep the
// one-thread-per-column sweeps.
bool thomas_chunks(const fen_ctx *c)
{
    const bool d2 = c->solver == FEN_SOLVER_PN || c->solver == FEN_SOLVER_NN;
    return d2 ? c->ny <= 4096 : c->nz <= 1024;
}

// Doubles of the c1 table thomas_chunk_kernel reads.
size_t thomas_chunk_c1_count(fen_ctx *c)
{
    const ChunkPlan pl = chunk_plan(c->solver, c->dim == 2 ? c->ny : c->nz);
    const ChunkArgs a = chunk_args(c, pl);
    return pl.d2 ? (size_t)a.ncol * a.n : (size_t)a.ncol * (a.nch > 1 ? a.nch - 1 : 1);
}

void launch_thomas_chunk_c1(fen_ctx *c)
{
    const ChunkPlan pl = chunk_plan(c->solver, c->dim == 2 ? c->ny : c->nz);
    const ChunkArgs a = chunk_args(c, pl);
    const dim3 grid((unsigned)((a.ncol + 255) / 256));
    if (pl.d2) hipLaunchKernelGGL(thomas_c1_kernel, grid, dim3(256), 0, c->stream, a, c->d_c1);
    else hipLaunchKernelGGL(thomas_starts_kernel, grid, dim3(256), 0, c->stream, a, c->d_c1, pl.m);
}

void launch_thomas_chunks(fen_ctx *c)
{
    const ChunkPlan pl = chunk_plan(c->solver, c->dim == 2 ? c->ny : c->nz);
    const ChunkArgs a = chunk_args(c, pl);
    if (a.nch * pl.cw > pl.nt) throw std::runtime_error("tridiagonal column too long for its workgroup");
    const bool f32 = c->precision != FEN_FP64;
    const bool real = c->solver == FEN_SOLVER_NN || c->solver == FEN_SOLVER_NNN;
    prof_begin(c, K_THOMAS);
    if (pl.d2) {
        if (real) launch_chunks_n<double, 8, 1, 1, 1>(c, a);
        else launch_chunks_n<double2, 8, 1, 1, 1>(c, a);
    } else if (real) {
        if (pl.cw == 16) launch_chunks_n<double, 16, 16, 2, 0>(c, a);
        else launch_chunks_n<double, 16, 8, 2, 0>(c, a);
    } else if (f32) {
        if (pl.m == 8) launch_chunks_n<float2, 8, 8, 3, 0>(c, a);
        else launch_chunks_n<float2, 16, 8, 1, 0>(c, a);
    } else {
        if (pl.m == 8) launch_chunks_n<double2, 8, 8, 3, 0>(c, a);
        else launch_chunks_n<double2, 16, 8, 1, 0>(c, a);
    }
    // columns read and written once
    prof_end(c, K_THOMAS, 2.0 * (real ? 8.0 : (f32 ? 8.0 : 16.0)) * (double)a.ncol * a.n);
}

}  // namespace fen
