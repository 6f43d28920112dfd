// adjoint.hip -- discrete adjoint of the FP64 time step (3-D, triply
// periodic, ppp, constant density and viscosity, fixed dt).  No counterpart
// in the reference: it differentiates navier_stokes_solver
// (src/navier_stokes.f90:50-136) as this library computes it.
//
// One forward step maps (u, p, dv_o) -> (u', p', dv_o'):
//   dv  = adv(u) + mu lap(u) / rho                 (advection in flux form)
//   u*  = u + dt (-G p / rho + A dv + B dv_o)       dv_o' = dv
//   phi = S (rho/dt) D u*                           (S: the FFT Poisson solve)
//   u'  = u* - (dt/rho) G phi                       p' = p + phi
// with D the MAC divergence, G the gradient (G^T = -D on the periodic grid)
// and S symmetric.  Its transpose, given (ub', pb', dvob'):
//   rb   = S (pb' + (dt/rho) D ub')       (the adjoint of the solve's right-hand side)
//   ub*  = ub' - (rho/dt) G rb
//   pb   = pb' + (dt/rho) D ub*
//   dvb  = dt A ub* + dvob'              dvob = dt B ub*
//   ub   = ub* + J_adv(u)^T dvb + (mu/rho) lap(dvb)
// J_adv^T is evaluated in gather form from the six advective fluxes
//   Qxx(i) = (u_i + u_{i+1})^2/4,  Rxy(i,j) = (u_{j} + u_{j+1})(v_i + v_{i+1})/4, ...
// each used by two momentum equations with opposite signs.  The adjoint of
// the forward state is needed at every step: a run is recorded with
// checkpoints every K steps and each segment is recomputed before its
// backward sweep.  Adjoint arrays are interior-sized (nx*ny*nz), i fastest;
// the recorded states are ghosted with their periodic images in place.
#include <algorithm>
#include <stdexcept>
#include <utility>
#include <vector>

#include "fen_internal.hpp"
#include "host_copy.hpp"

namespace fen {

namespace {

struct AdjDims {
    int nx, ny, nz;
    long gx, gxy;
    __device__ long q(int i, int j, int k) const { return i + (long)nx * (j + (long)ny * k); }   // 0-based
};

struct AdjStepArgs {
    const double *u, *v, *w;      // recorded state (ghosted)
    const double *ub[3], *dvo[3]; // ub', dvob'
    const double *psi;            // rb = S (pb' + (dt/rho) D ub')
    double *pb;                   // in pb', out pb
    double *ub_out[3], *dvo_out[3];
    double id, id2, mu_rho, s, dt_rho, dtA, dtB;   // s = rho/dt
    int nbx, nby, kb;             // tiles along x, y; planes per march
};

// One transposed step after its solve:
//   ub* = ub' - (rho/dt) G rb, pb += (dt/rho) D ub*, dvb = dtA ub* + dvob',
//   dvob = dtB ub*, ub = ub* + J_adv^T dvb + (mu/rho) lap(dvb), gathered per face,
// as a k-march: a 64x4 tile of cells walks kb planes of z with planes k-1, k,
// k+1 of u, v, w (ghosted, images in place) and of dvb in an LDS ring, and x,
// y of ub* at planes k, k+1 (their divergence; z is carried).  Plane k+2 is
// loaded into registers while plane k is computed.  A thread's first tile
// element is its own cell, so what the cell needs of ub* stays in registers;
// the second, for the first 140 threads, is one of the halo's.
// It moves 18 words per cell at 3.8 TB/s, 0.8 of a device copy: HBM and the
// march's own chain (two barriers per plane, one row per thread, a halo of 0.55
// of the tile from the L2 that neighbouring workgroups share) bound it together.
// 80 us at 128^3, 88 with tiles dealt round the XCDs; with ub* and dvb formed by a kernel of their own,
// 12 words more, 60 + 61.
constexpr int kMX = 64, kMY = 4;
constexpr int kMLX = kMX + 2, kMN = kMLX * (kMY + 2);      // haloed tile
constexpr int kMHalo = 2 * kMLX + 2 * kMY;

__global__ __launch_bounds__(kMX * kMY) void adj_step_kernel(AdjDims d, AdjStepArgs a)
{
    __shared__ double lds[6 * 3 * kMN];   // [field u v w A B E][slot][tile]
    __shared__ double star[2 * 2 * kMN];  // [ub*, vb*][slot][tile]
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int i0 = bid % a.nbx * kMX, j0 = bid / a.nbx % a.nby * kMY, k0 = bid / (a.nbx * a.nby) * a.kb;
    const int kend = min(k0 + a.kb, d.nz);
    const int tx = threadIdx.x % kMX, ty = threadIdx.x / kMX;
    const int i = i0 + tx, j = j0 + ty;
    const bool active = i < d.nx && j < d.ny;
    const int nx = d.nx, ny = d.ny, nz = d.nz;
    const int c = (ty + 1) * kMLX + tx + 1;
    // the tile elements: position in the tile, offsets in a ghosted and in an
    // interior (wrapped) plane, and of the interior neighbours above along x, y.
    // Past the grid clamped to the last ghost (values no active cell reads)
    const int h = (int)threadIdx.x;
    const bool halo = h < kMHalo;
    int hi = 0, hj = 0;
    if (h < 2 * kMLX) {
        hi = h % kMLX;
        hj = h < kMLX ? 0 : kMY + 1;
    } else if (halo) {
        hi = h < 2 * kMLX + kMY ? 0 : kMX + 1;
        hj = (h - 2 * kMLX) % kMY + 1;
    }
    const int pos[2] = {c, hi + kMLX * hj};
    int og[2], oq[2], ox[2], oy[2];
#pragma unroll
    for (int m = 0; m < 2; m++) {
        const int ii = min(i0 - 1 + pos[m] % kMLX, nx), jj = min(j0 - 1 + pos[m] / kMLX, ny);
        const int iq = ii < 0 ? nx - 1 : (ii == nx ? 0 : ii), jq = jj < 0 ? ny - 1 : (jj == ny ? 0 : jj);
        og[m] = (ii + 1) + (int)d.gx * (jj + 1);
        oq[m] = iq + nx * jq;
        ox[m] = (iq + 1 == nx ? 0 : iq + 1) + nx * jq;
        oy[m] = iq + nx * (jq + 1 == ny ? 0 : jq + 1);
    }
    const long plane = (long)nx * ny;
    double raw[2][13];
    auto fetch = [&](int kk) {   // plane kk in [-1, nz]
        const int kw = kk < 0 ? nz - 1 : (kk == nz ? 0 : kk);
        const long kg = d.gxy * (kk + 1), kq = plane * kw, kz = plane * (kw + 1 == nz ? 0 : kw + 1);
#pragma unroll
        for (int m = 0; m < 2; m++) {
            if (m == 1 && !halo) continue;
            raw[m][0] = a.u[kg + og[m]];
            raw[m][1] = a.v[kg + og[m]];
            raw[m][2] = a.w[kg + og[m]];
#pragma unroll
            for (int f = 0; f < 3; f++) {
                raw[m][3 + f] = a.ub[f][kq + oq[m]];
                raw[m][6 + f] = a.dvo[f][kq + oq[m]];
            }
            raw[m][9] = a.psi[kq + oq[m]];
            raw[m][10] = a.psi[kq + ox[m]];
            raw[m][11] = a.psi[kq + oy[m]];
            raw[m][12] = a.psi[kz + oq[m]];
        }
    };
    // the fetched plane into ring slot `slot` and star slot `ss`; own: ub* of the thread's cell
    auto commit = [&](int slot, int ss, double (&own)[3]) {
#pragma unroll
        for (int m = 0; m < 2; m++) {
            if (m == 1 && !halo) continue;
            const int e = pos[m];
#pragma unroll
            for (int f = 0; f < 3; f++) {
                const double st = raw[m][3 + f] - a.s * ((raw[m][10 + f] - raw[m][9]) * a.id);
                lds[(f * 3 + slot) * kMN + e] = raw[m][f];
                lds[((3 + f) * 3 + slot) * kMN + e] = a.dtA * st + raw[m][6 + f];
                if (f < 2) star[(f * 2 + ss) * kMN + e] = st;
                if (m == 0) own[f] = st;
            }
        }
    };
    double below[3], here[3], above[3];   // ub* of the thread's cell at k - 1, k, k + 1
    fetch(k0 - 1);
    commit(0, 0, below);   // (star slot 0 is written again for k0, each element by the same thread)
    fetch(k0);
    commit(1, 0, here);
    fetch(k0 + 1);
    int sm = 0, sc = 1, sn = 2, ss = 0;
    const double id = a.id;
    for (int k = k0; k < kend; k++) {
        commit(sn, ss ^ 1, above);   // plane k + 1
        __syncthreads();
        if (k + 2 <= nz && k + 2 <= kend) fetch(k + 2);
        if (active) {
            const long q = d.q(i, j, k);
            const double sxm = star[ss * kMN + c - 1], sym = star[(2 + ss) * kMN + c - kMLX];
            const double div = ((here[0] - sxm) * id + (here[1] - sym) * id) + (here[2] - below[2]) * id;
            a.pb[q] = a.pb[q] + a.dt_rho * div;
#pragma unroll
            for (int f = 0; f < 3; f++) a.dvo_out[f][q] = a.dtB * here[f];
            auto at = [&](int f, int di, int dj, int dk) {
                const int sl = dk < 0 ? sm : (dk > 0 ? sn : sc);
                return lds[(f * 3 + sl) * kMN + c + dj * kMLX + di];
            };
            auto U = [&](int di, int dj, int dk) { return at(0, di, dj, dk); };
            auto V = [&](int di, int dj, int dk) { return at(1, di, dj, dk); };
            auto W = [&](int di, int dj, int dk) { return at(2, di, dj, dk); };
            auto A = [&](int di, int dj, int dk) { return at(3, di, dj, dk); };
            auto B = [&](int di, int dj, int dk) { return at(4, di, dj, dk); };
            auto E = [&](int di, int dj, int dk) { return at(5, di, dj, dk); };
            // flux adjoints at offsets from (i, j, k)
            auto Qxx = [&](int di, int dj, int dk) { return (A(di + 1, dj, dk) - A(di, dj, dk)) * id; };
            auto Qyy = [&](int di, int dj, int dk) { return (B(di, dj + 1, dk) - B(di, dj, dk)) * id; };
            auto Qzz = [&](int di, int dj, int dk) { return (E(di, dj, dk + 1) - E(di, dj, dk)) * id; };
            auto Rxy = [&](int di, int dj, int dk) {
                return (A(di, dj + 1, dk) - A(di, dj, dk)) * id + (B(di + 1, dj, dk) - B(di, dj, dk)) * id;
            };
            auto Rxz = [&](int di, int dj, int dk) {
                return (A(di, dj, dk + 1) - A(di, dj, dk)) * id + (E(di + 1, dj, dk) - E(di, dj, dk)) * id;
            };
            auto Ryz = [&](int di, int dj, int dk) {
                return (B(di, dj, dk + 1) - B(di, dj, dk)) * id + (E(di, dj + 1, dk) - E(di, dj, dk)) * id;
            };
            auto lap = [&](int f) {
                const double c0 = at(f, 0, 0, 0);
                return ((at(f, 1, 0, 0) - 2.0 * c0 + at(f, -1, 0, 0)) + (at(f, 0, 1, 0) - 2.0 * c0 + at(f, 0, -1, 0)) +
                        (at(f, 0, 0, 1) - 2.0 * c0 + at(f, 0, 0, -1))) * a.id2;
            };
            const double u0 = U(0, 0, 0), v0 = V(0, 0, 0), w0 = W(0, 0, 0);
            double gu = Qxx(0, 0, 0) * 0.5 * (u0 + U(1, 0, 0)) + Qxx(-1, 0, 0) * 0.5 * (U(-1, 0, 0) + u0);
            gu += Rxy(0, 0, 0) * 0.25 * (V(1, 0, 0) + v0) + Rxy(0, -1, 0) * 0.25 * (V(1, -1, 0) + V(0, -1, 0));
            gu += Rxz(0, 0, 0) * 0.25 * (W(1, 0, 0) + w0) + Rxz(0, 0, -1) * 0.25 * (W(1, 0, -1) + W(0, 0, -1));
            double gv = Qyy(0, 0, 0) * 0.5 * (v0 + V(0, 1, 0)) + Qyy(0, -1, 0) * 0.5 * (V(0, -1, 0) + v0);
            gv += Rxy(0, 0, 0) * 0.25 * (U(0, 1, 0) + u0) + Rxy(-1, 0, 0) * 0.25 * (U(-1, 1, 0) + U(-1, 0, 0));
            gv += Ryz(0, 0, 0) * 0.25 * (W(0, 1, 0) + w0) + Ryz(0, 0, -1) * 0.25 * (W(0, 1, -1) + W(0, 0, -1));
            double gw = Qzz(0, 0, 0) * 0.5 * (w0 + W(0, 0, 1)) + Qzz(0, 0, -1) * 0.5 * (W(0, 0, -1) + w0);
            gw += Rxz(0, 0, 0) * 0.25 * (U(0, 0, 1) + u0) + Rxz(-1, 0, 0) * 0.25 * (U(-1, 0, 1) + U(-1, 0, 0));
            gw += Ryz(0, 0, 0) * 0.25 * (V(0, 0, 1) + v0) + Ryz(0, -1, 0) * 0.25 * (V(0, -1, 1) + V(0, -1, 0));
            a.ub_out[0][q] = here[0] + gu + a.mu_rho * lap(3);
            a.ub_out[1][q] = here[1] + gv + a.mu_rho * lap(4);
            a.ub_out[2][q] = here[2] + gw + a.mu_rho * lap(5);
        }
        __syncthreads();   // every read of slot sm precedes the next commit into it
        const int t = sm;
        sm = sc; sc = sn; sn = t;
        ss ^= 1;
#pragma unroll
        for (int f = 0; f < 3; f++) {
            below[f] = here[f];
            here[f] = above[f];
        }
    }
}

}  // namespace

// Recorded run: checkpoints of the full state every `every` steps, plus the
// final state; segment buffer of the velocity at the start of each step.
struct AdjointTape {
    int nsteps = 0, every = 0, step0 = 0;
    double dt = 0.0, dt_o = 0.0;
    std::vector<double *> ckpt;    // [u v w p](ghosted) [dvo x3](interior), one block per checkpoint
    double *final_state = nullptr;
    std::vector<double *> seg;     // every x [u v w](ghosted)
    double *work = nullptr;        // 14 interior arrays: adjoint state [ub x3][pb][dvob x3], next [ub x3][dvob x3], rb
};

namespace {

size_t ckpt_len(const fen_ctx *c) { return 4 * c->n_ghost + 3 * c->n_int; }

void save_state(fen_ctx *c, double *dst)
{
    const size_t ng = c->n_ghost * sizeof(double), ni = c->n_int * sizeof(double);
    for (int d = 0; d < 3; d++)
        FEN_HIP_CHECK(hipMemcpyAsync(dst + d * c->n_ghost, c->d_u[d], ng, hipMemcpyDeviceToDevice, c->stream));
    FEN_HIP_CHECK(hipMemcpyAsync(dst + 3 * c->n_ghost, c->d_p, ng, hipMemcpyDeviceToDevice, c->stream));
    for (int d = 0; d < 3; d++)
        FEN_HIP_CHECK(hipMemcpyAsync(dst + 4 * c->n_ghost + d * c->n_int, c->d_dvo[d], ni, hipMemcpyDeviceToDevice,
                                     c->stream));
}

void load_state(fen_ctx *c, const double *src)
{
    const size_t ng = c->n_ghost * sizeof(double), ni = c->n_int * sizeof(double);
    for (int d = 0; d < 3; d++)
        FEN_HIP_CHECK(hipMemcpyAsync(c->d_u[d], src + d * c->n_ghost, ng, hipMemcpyDeviceToDevice, c->stream));
    FEN_HIP_CHECK(hipMemcpyAsync(c->d_p, src + 3 * c->n_ghost, ng, hipMemcpyDeviceToDevice, c->stream));
    for (int d = 0; d < 3; d++)
        FEN_HIP_CHECK(hipMemcpyAsync(c->d_dvo[d], src + 4 * c->n_ghost + d * c->n_int, ni, hipMemcpyDeviceToDevice,
                                     c->stream));
}

double *dalloc(size_t n)
{
    void *p = nullptr;
    FEN_HIP_CHECK(hipMalloc(&p, n * sizeof(double)));
    return static_cast<double *>(p);
}

AdjDims dims(const fen_ctx *c) { return AdjDims{c->nx, c->ny, c->nz, c->box.gx, c->box.gxy}; }

// Planes per march: 16 (18 are formed for them) where that gives two
// workgroups per CU, as many as its LDS holds; shorter ones on smaller grids,
// down to 4.
int march_planes(const fen_ctx *c, long tiles)
{
    int kb = 16;
    while (kb > 4 && tiles * ((c->nz + kb - 1) / kb) < 2L * c->num_cu) kb /= 2;
    return kb;
}

// One adjoint step at the recorded state `st` ([u v w] ghosted); ub and dvo
// become the arrays of ub_out and dvo_out, and those the old ones.
void adjoint_step(fen_ctx *c, AdjointTape *t, const double *st, double **ub, double *pb, double **dvo, double **ub_out,
                  double **dvo_out)
{
    double *r = t->work + 13 * c->n_int;
    const AdjDims d = dims(c);
    const double rho = c->density, dt = t->dt;
    const double id = 1.0 / c->delta;
    const double A = 1.0 + 0.5 * dt / t->dt_o, B = -(0.5 * dt / t->dt_o);
    // r = S (pb' + (dt/rho) D ub'): the adjoint of the solve's right-hand side,
    // formed by the x transform's loads (a pass of its own, written and read
    // back, took 17 + 10 us at 128^3 against 20)
    const long sx = c->nx, sy = (long)c->nx * c->ny;
    const bool plane = plane_pass(c);
    if (plane) {
        launch_plane_adj(c, ub, pb, dt / rho);
    } else {
        launch_adj_r2c(c, ub, pb, dt / rho);
        launch_y_fft<double>(c, -1, 1.0);
    }
    launch_z_solve<double>(c, 1.0 / (double)(float)((long)c->nx * c->ny * c->nz));
    if (!plane) launch_y_fft<double>(c, +1, 1.0);
    launch_c2r<double>(c, r, 0, sx, sy, false, AxisCopies{});
    AdjStepArgs a{};
    a.u = st; a.v = st + c->n_ghost; a.w = st + 2 * c->n_ghost;
    for (int k = 0; k < 3; k++) {
        a.ub[k] = ub[k]; a.dvo[k] = dvo[k];
        a.ub_out[k] = ub_out[k]; a.dvo_out[k] = dvo_out[k];
    }
    a.psi = r;
    a.pb = pb;
    a.id = id;
    a.id2 = 1.0 / (c->delta * c->delta);
    a.mu_rho = c->viscosity / rho;
    a.s = rho / dt;
    a.dt_rho = dt / rho;
    a.dtA = dt * A;
    a.dtB = dt * B;
    a.nbx = (c->nx + kMX - 1) / kMX;
    a.nby = (c->ny + kMY - 1) / kMY;
    const long tiles = (long)a.nbx * a.nby;
    a.kb = march_planes(c, tiles);
    hipLaunchKernelGGL(adj_step_kernel, dim3((unsigned)(tiles * ((c->nz + a.kb - 1) / a.kb))), dim3(kMX * kMY), 0, c->stream, d, a);
    for (int k = 0; k < 3; k++) {
        std::swap(ub[k], ub_out[k]);
        std::swap(dvo[k], dvo_out[k]);
    }
}

}  // namespace

void adjoint_free(fen_ctx *c)
{
    AdjointTape *t = c->tape;
    if (!t) return;
    for (double *p : t->ckpt) (void)hipFree(p);
    for (double *p : t->seg) (void)hipFree(p);
    if (t->final_state) (void)hipFree(t->final_state);
    if (t->work) (void)hipFree(t->work);
    delete t;
    c->tape = nullptr;
}

// A tape for nseg checkpoints and segments of `every` states that holds the
// blocks of the context's last one, 50 to 270 MB each at 128^3: the first
// gradient of a context (60 steps, every 20) takes 32.4 ms, the next 29.3; with
// every record freeing and allocating them 37.6 and 42.5.  Blocks beyond these
// counts are given back.
static AdjointTape *reuse_tape(fen_ctx *c, int nseg, int every)
{
    if (!c->tape) c->tape = new AdjointTape();
    AdjointTape *t = c->tape;
    auto keep = [](std::vector<double *> &v, size_t n) {
        for (; v.size() > n; v.pop_back()) (void)hipFree(v.back());
    };
    keep(t->ckpt, (size_t)nseg);
    keep(t->seg, (size_t)every);
    return t;
}

bool adjoint_recorded(const fen_ctx *c) { return c->tape && c->tape->nsteps > 0; }

const char *adjoint_unsupported(const fen_ctx *c)
{
    if (c->precision != FEN_FP64) return "the adjoint is provided for FP64 contexts";
    if (c->dim != 3 || c->solver != FEN_SOLVER_PPP) return "the adjoint needs a 3-D triply periodic grid";
    if (c->has_source) return "the adjoint does not include a source term";
    if (c->constant_cfl) return "the adjoint needs a fixed dt (constant_CFL off)";
    return nullptr;
}

void adjoint_record(fen_ctx *c, int step0, int nsteps, int every, double dt)
{
    const int nseg = (nsteps + every - 1) / every;
    AdjointTape *t = reuse_tape(c, nseg, every);
    t->nsteps = 0;   // nothing recorded if this fails
    auto more = [&](std::vector<double *> &v, size_t n, size_t len) {
        while (v.size() < n) v.push_back(dalloc(len));
    };
    more(t->ckpt, (size_t)nseg, ckpt_len(c));
    if (!t->final_state) t->final_state = dalloc(ckpt_len(c));
    t->every = every;
    t->step0 = step0;
    t->dt = dt;
    t->dt_o = c->dt_o;
    for (int s = 0; s < nsteps; s += every) {
        save_state(c, t->ckpt[s / every]);
        run_fp64(c, std::min(every, nsteps - s), dt);
    }
    save_state(c, t->final_state);
    FEN_HIP_CHECK(hipStreamSynchronize(c->stream));
    t->nsteps = nsteps;
}

void adjoint_backward(fen_ctx *c, const double *seed[3], double *grad[3], double *grad_p)
{
    AdjointTape *t = c->tape;
    const size_t n = c->n_int;
    if (!t->work) t->work = dalloc(14 * n);
    while ((int)t->seg.size() < std::min(t->every, t->nsteps)) t->seg.push_back(dalloc(3 * c->n_ghost));
    double *ub[3] = {t->work, t->work + n, t->work + 2 * n}, *pb = t->work + 3 * n;
    double *dvo[3] = {t->work + 4 * n, t->work + 5 * n, t->work + 6 * n};
    double *ub2[3] = {t->work + 7 * n, t->work + 8 * n, t->work + 9 * n};
    double *dvo2[3] = {t->work + 10 * n, t->work + 11 * n, t->work + 12 * n};
    for (int d = 0; d < 3; d++) queue_to_device(c->stream, ub[d], seed[d], n);
    FEN_HIP_CHECK(hipMemsetAsync(pb, 0, 4 * n * sizeof(double), c->stream));   // pb and dvo
    const double dt_o_saved = c->dt_o;
    c->dt_o = t->dt_o;
    const int nseg = (t->nsteps + t->every - 1) / t->every;
    for (int sg = nseg - 1; sg >= 0; sg--) {
        const int first = sg * t->every, len = std::min(t->every, t->nsteps - first);
        load_state(c, t->ckpt[sg]);
        // the segment's states, each formed straight into its slot (the
        // state after the segment's last step is not needed)
        states_fp64(c, t->dt, len, t->seg.data());
        for (int s = len - 1; s >= 0; s--) adjoint_step(c, t, t->seg[s], ub, pb, dvo, ub2, dvo2);
    }
    for (int d = 0; d < 3; d++) queue_to_host(c->stream, grad[d], ub[d], n);
    if (grad_p) queue_to_host(c->stream, grad_p, pb, n);
    load_state(c, t->final_state);   // leave the context at the end of the recorded run
    c->dt_o = dt_o_saved;
    c->checks_valid = false;
    FEN_HIP_CHECK(hipStreamSynchronize(c->stream));
}

}  // namespace fen
