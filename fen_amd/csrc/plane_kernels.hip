// plane_kernels.hip -- the x and y transforms of the triply periodic and the
// channel solver (ppp, ppn) on planes small enough for LDS: one workgroup
// takes a whole z plane, so the right-hand side is transformed along x and y
// (and back to phi along y and x) without the half-transformed spectrum going
// through memory.
//
// Forward: row pairs as complex lines through the x FFT; each kx column is
// unpacked from the packed lines in LDS straight into the y FFT's registers.
// Backward: the same steps in reverse.  Half spectrum [kx][k][j] and
// arithmetic are the separate passes'.
//
// There are NX/2 + 1 columns and threads for NX/2: the last one waits in an LDS
// line of its own until the first wave has transformed its other columns.  (The
// columns 0 and NX/2 are real sequences in y and could share one complex line,
// but column NX/2 then takes on the round-off of column 0, which is far larger in
// a solution: up to 1.39 times the error of a solve, at 16 x 64 x 32.  A line of
// its own costs 32 x 128 x 32 1.6 us per step, the others at most 0.6; as NY/8
// more threads it cost 128 x 64 x 128 14, one workgroup per CU instead of two.)
//
// What bounds it: the latency of one workgroup's chain, load to store; the
// separate passes pay it twice each way, with a launch between.  Us per step,
// separate passes -> planes, FP64 (FP32): 32^3 27.2 -> 22.7 (25.1 -> 22.6),
// 64^3 35.5 -> 32.4 (30.8 -> 27.7), 64 x 64 x 256 72 -> 60 (51 -> 44).
#include <stdexcept>

#include "fen_internal.hpp"
#include "fft_device.hpp"
#include "rhs_device.hpp"

namespace fen {

namespace {

template <class R> struct PlaneArgs {
    using C = typename Cplx<R>::type;
    // forward (rhs_load's)
    const R *u, *v, *w, *p;
    C *spec;
    const C *twx, *twy;
    Box b;
    double id, rho, dt, scale, postx, posty;
    long sx, sy;
    int gl, nz;
    // backward
    R *out;
    AxisCopies copies;
    int want_sum;
    double *part;
};

template <int NX, int NY> constexpr int plane_threads() { return NX * NY / 16; }
template <int NX, int NY> constexpr int plane_lds()
{
    constexpr int a = NY / 2 * lds_line<NX>(), b = NX / 2 * lds_line<NY>();
    return a > b ? a : b;
}

template <class R, int NX, int NY, int MODE>
__global__ __launch_bounds__((plane_threads<NX, NY>())) void plane_fwd_kernel(PlaneArgs<R> a)
{
    using C = typename Cplx<R>::type;
    constexpr int TX = NX / 8, TY = NY / 8, LX = lds_line<NX>(), LY = lds_line<NY>();
    __shared__ C buf[plane_lds<NX, NY>()], last[LY];   // last: column NX/2
    __shared__ C twx[NX], twy[NY];
    load_twiddles<NX>(twx, a.twx);   // first read after the first stage's barrier
    load_twiddles<NY>(twy, a.twy);
    const int k = blockIdx.x + 1;
    const int l = threadIdx.x / TX, t = threadIdx.x % TX;
    C v[8];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int j = 2 * l + h + 1;
        R f[8][7];   // the row's loads, all issued before the first is used
#pragma unroll
        for (int q = 0; q < 8; q++) rhs_load<R, MODE, 1>(a, f[q], t + q * TX + 1, j, k);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const double val = rhs_value<R, MODE, 1>(a, f[q]);
            if (h == 0) v[q].x = (R)val;
            else v[q].y = (R)val;
        }
    }
    C *line = buf + l * LX;
    fft_regs<NX, -1>(v, line, t, twx);
#pragma unroll
    for (int q = 0; q < 8; q++) line[lds_pad(t + q * TX)] = v[q];
    __syncthreads();
    // column c: rows 2l, 2l + 1 of every pair at kx = c
    const int c = threadIdx.x / TY, s = threadIdx.x % TY;
    const R half = R(0.5), postx = (R)a.postx;
    auto unpack = [&](int kx, int j) {
        const C *ln = buf + (j >> 1) * LX;
        const C zk = ln[lds_pad(kx)], zn = ln[lds_pad((NX - kx) & (NX - 1))];
        C x;
        if (j & 1) x = C{(zk.y + zn.y) * half, (zn.x - zk.x) * half};
        else x = C{(zk.x + zn.x) * half, (zk.y - zn.y) * half};
        return C{x.x * postx, x.y * postx};
    };
#pragma unroll
    for (int q = 0; q < 8; q++) v[q] = unpack(c, s + q * TY);
    if (c == 0) {
#pragma unroll
        for (int q = 0; q < 8; q++) last[lds_pad(s + q * TY)] = unpack(NX / 2, s + q * TY);
    }
    __syncthreads();   // every read of the packed lines precedes the y stages' writes
    auto put = [&](int kx) {
        C *out = a.spec + ((long)kx * a.nz + (k - 1)) * NY;
#pragma unroll
        for (int q = 0; q < 8; q++)
            out[s + q * TY] = C{(R)((double)v[q].x * a.posty), (R)((double)v[q].y * a.posty)};
    };
    fft_regs<NY, -1>(v, buf + c * LY, s, twy);
    put(c);
    if (c == 0) {   // the threads of column 0, all in the first wave
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] = last[lds_pad(s + q * TY)];
        fft_sync<1>();
        fft_regs<NY, -1, 1>(v, last, s, twy);
        put(NX / 2);
    }
}

template <class R, int NX, int NY>
__global__ __launch_bounds__((plane_threads<NX, NY>())) void plane_bwd_kernel(PlaneArgs<R> a)
{
    using C = typename Cplx<R>::type;
    constexpr int TX = NX / 8, TY = NY / 8, LX = lds_line<NX>(), LY = lds_line<NY>(), NT = plane_threads<NX, NY>();
    __shared__ C buf[plane_lds<NX, NY>()], last[LY];   // last: column NX/2
    __shared__ C twx[NX], twy[NY];
    load_twiddles<NX>(twx, a.twx);
    load_twiddles<NY>(twy, a.twy);
    const int k = blockIdx.x;
    const int c = threadIdx.x / TY, s = threadIdx.x % TY;
    const C *in = a.spec + ((long)c * a.nz + k) * NY;
    C v[8], vl[8];
#pragma unroll
    for (int q = 0; q < 8; q++) v[q] = in[s + q * TY];
    if (c == 0) {
        const C *il = a.spec + ((long)(NX / 2) * a.nz + k) * NY;
#pragma unroll
        for (int q = 0; q < 8; q++) vl[q] = il[s + q * TY];
    }
    C *col = buf + c * LY;
    fft_regs<NY, 1>(v, col, s, twy);
#pragma unroll
    for (int q = 0; q < 8; q++) col[lds_pad(s + q * TY)] = v[q];
    if (c == 0) {   // the threads of column 0, all in the first wave
        fft_regs<NY, 1, 1>(vl, last, s, twy);
#pragma unroll
        for (int q = 0; q < 8; q++) last[lds_pad(s + q * TY)] = vl[q];
    }
    __syncthreads();
    const int l = threadIdx.x / TX, t = threadIdx.x % TX;
    const int r0 = lds_pad(2 * l), r1 = lds_pad(2 * l + 1);
#pragma unroll
    for (int q = 0; q < 8; q++) {
        const int kx = t + q * TX;
        const int m = kx <= NX / 2 ? kx : NX - kx;
        const C *cl = m == NX / 2 ? last : buf + m * LY;
        const C x1 = cl[r0], x2 = cl[r1];
        if (kx == 0 || kx == NX / 2) v[q] = C{x1.x, x2.x};   // Im of bins 0 and NX/2 ignored
        else if (kx < NX / 2) v[q] = C{x1.x - x2.y, x1.y + x2.x};
        else v[q] = C{x1.x + x2.y, x2.x - x1.y};
    }
    __syncthreads();   // every read of the columns precedes the x stages' writes
    fft_regs<NX, 1>(v, buf + l * LX, t, twx);
    double acc = 0.0;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int j = 2 * l + h;
        int jd[3], kd[3], nj = 1, nk = 1;
        jd[0] = j + a.gl;
        kd[0] = k + a.gl;
        if (a.copies.any()) {
            nj = copy_rows(j + 1, NY, a.copies.y, jd);
            nk = copy_rows(k + 1, a.nz, a.copies.z, kd);
        }
        for (int dk = 0; dk < nk; dk++)
            for (int dj = 0; dj < nj; dj++) {
                R *orow = a.out + a.gl + a.sx * jd[dj] + a.sy * kd[dk];
#pragma unroll
                for (int q = 0; q < 8; q++) orow[t + q * TX] = h ? v[q].y : v[q].x;
                if (a.copies.x) {
                    if (t == 0) orow[NX] = h ? v[0].y : v[0].x;
                    if (t == TX - 1) orow[-1] = h ? v[7].y : v[7].x;
                }
            }
#pragma unroll
        for (int q = 0; q < 8; q++) acc += (double)(h ? v[q].y : v[q].x);
    }
    if (a.want_sum) {   // fft_regs has finished every read of buf: reuse it
        double *red = reinterpret_cast<double *>(buf);
        red[threadIdx.x] = acc;
        __syncthreads();
        for (int w = NT / 2; w > 0; w >>= 1) {
            if ((int)threadIdx.x < w) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + w];
            __syncthreads();
        }
        if (threadIdx.x == 0) a.part[blockIdx.x] = red[0];
    }
}

#define FEN_PLANE_CASE(NX, NY) case NX * 1024 + NY: FEN_PLANE_RUN(NX, NY); break;
#define FEN_PLANE                                                                        \
    switch (c->nx * 1024 + c->ny) {                                                      \
    FEN_PLANE_CASE(16, 64) FEN_PLANE_CASE(16, 128)                                       \
    FEN_PLANE_CASE(32, 32) FEN_PLANE_CASE(32, 64) FEN_PLANE_CASE(32, 128)                \
    FEN_PLANE_CASE(64, 16) FEN_PLANE_CASE(64, 32) FEN_PLANE_CASE(64, 64)                 \
    FEN_PLANE_CASE(64, 128)                                                              \
    FEN_PLANE_CASE(128, 16) FEN_PLANE_CASE(128, 32) FEN_PLANE_CASE(128, 64)              \
    default: throw std::runtime_error("plane transform length");                         \
    }

template <class R> PlaneArgs<R> plane_args(fen_ctx *c)
{
    using C = typename Cplx<R>::type;
    PlaneArgs<R> a{};
    a.spec = as<C>(c->d_spec);
    a.twx = as<C>(c->d_twx);
    a.twy = as<C>(c->d_twy);
    a.b = c->box;
    a.id = 1.0 / c->delta;
    a.nz = c->nz;
    return a;
}

template <class R, int MODE> void launch_fwd(fen_ctx *c, const PlaneArgs<R> &a, double words)
{
    prof_begin(c, K_DIV_R2C);
#define FEN_PLANE_RUN(NX, NY) \
    hipLaunchKernelGGL((plane_fwd_kernel<R, NX, NY, MODE>), dim3((unsigned)c->nz), dim3(plane_threads<NX, NY>()), 0, c->stream, a)
    FEN_PLANE
#undef FEN_PLANE_RUN
    prof_end(c, K_DIV_R2C, (words + 1.0) * sizeof(R) * c->n_int);
}

}  // namespace

bool plane_pass(const fen_ctx *c)
{
    // One workgroup per plane, 16 points per thread.  Under one wave a plane is
    // slower than its passes (32 x 16 x 32: 25.7 -> 32 us per step); up to four
    // waves it is faster at every nz; eight waves need planes for half the CUs
    // (128 x 64, FP64: 64 planes 47.1 -> 47.7, 128 planes 70 -> 64.6, 512
    // planes 209 -> 191); with sixteen (128 x 128) one workgroup fills a CU and few
    // planes leave the others idle (32 planes 48 -> 68; 128: the passes 67 us
    // either way; 256: 201 -> 194).
    if (c->dim != 3 || (c->solver != FEN_SOLVER_PPP && c->solver != FEN_SOLVER_PPN)) return false;
    // One block sum per plane: at most the 32768 that the allocation-free
    // solve's fixed scratch holds, so that it takes every grid it would without.
    const long m = (long)c->nx * c->ny;
    if (c->nz > 32768) return false;
    return c->nx >= 16 && c->nx <= 128 && c->ny >= 16 && c->ny <= 128 && m >= 1024 && (m <= 4096 || (m <= 8192 && c->nz >= 128));
}

template <class R>
void launch_plane_fwd(fen_ctx *c, const R *const *vel, const R *direct, long sx, long sy, int gl, double rho, double dt,
                      double postx, double posty)
{
    PlaneArgs<R> a = plane_args<R>(c);
    a.rho = rho;
    a.dt = dt;
    a.postx = postx;
    a.posty = posty;
    if (vel) {
        a.u = vel[0]; a.v = vel[1]; a.w = vel[2];
        launch_fwd<R, 0>(c, a, 3.0);
    } else {
        a.u = direct; a.sx = sx; a.sy = sy; a.gl = gl;
        launch_fwd<R, 1>(c, a, 1.0);
    }
}

void launch_plane_adj(fen_ctx *c, const double *const *vel, const double *p, double scale)
{
    PlaneArgs<double> a = plane_args<double>(c);
    a.u = vel[0]; a.v = vel[1]; a.w = vel[2];
    a.p = p;
    a.scale = scale;
    a.postx = a.posty = 1.0;
    launch_fwd<double, 2>(c, a, 4.0);
}

template <class R>
void launch_plane_bwd(fen_ctx *c, R *phi, int gl, long sx, long sy, AxisCopies copies, double *part)
{
    PlaneArgs<R> a = plane_args<R>(c);
    a.out = phi;
    a.gl = gl;
    a.sx = sx;
    a.sy = sy;
    a.copies = copies;
    a.want_sum = part ? 1 : 0;
    a.part = part;
    prof_begin(c, K_C2R);
#define FEN_PLANE_RUN(NX, NY) \
    hipLaunchKernelGGL((plane_bwd_kernel<R, NX, NY>), dim3((unsigned)c->nz), dim3(plane_threads<NX, NY>()), 0, c->stream, a)
    FEN_PLANE
#undef FEN_PLANE_RUN
    prof_end(c, K_C2R, 2.0 * sizeof(R) * c->n_int);
}

#define FEN_INSTANTIATE(R)                                                                                            \
    template void launch_plane_fwd<R>(fen_ctx *, const R *const *, const R *, long, long, int, double, double, double, \
                                      double);                                                                        \
    template void launch_plane_bwd<R>(fen_ctx *, R *, int, long, long, AxisCopies, double *);
FEN_INSTANTIATE(double)
FEN_INSTANTIATE(float)
#undef FEN_INSTANTIATE

}  // namespace fen
