// fused_kernels.hip -- step n's projection fused with step n+1's momentum
// (stencil_march.hpp): which grids take it, how they are cut, the launches.
#include <algorithm>
#include <stdexcept>
#include <type_traits>

#include "fen_internal.hpp"
#include "stencil_march.hpp"

namespace fen {

// x and y periodic for every field, z faces no-slip walls (the ghost rules
// the fused kernel evaluates itself): u, v, w Dirichlet, p and phi Neumann.
bool fused_z_walls(const fen_ctx *c)
{
    if (c->box.dim != 3 || c->img_vel != 3 || c->img_p != 3 || c->img_phi != 3) return false;
    for (int f : {FEN_FRONT, FEN_BACK}) {
        if (c->bc_type[FEN_U][f] != 1 || c->bc_type[FEN_V][f] != 1 || c->bc_type[FEN_W][f] != 1) return false;
        if (c->bc_type[FEN_P][f] != 2 || c->bc_type[FEN_PHI][f] != 2) return false;
    }
    return true;
}

// The general-wall form of the fused kernel (3-D FP64, no pending mean
// shift; the Neumann-direction grids npn and nnn): every axis of every
// state field is periodic on both faces, or Dirichlet/Neumann on both
// (the tile formation evaluates the ghost fill's rule chain).  Grids the
// two dedicated forms take are excluded.
bool fused_general_walls(const fen_ctx *c)
{
    if (c->box.dim != 3 || c->precision != FEN_FP64) return false;
    if (c->solver != FEN_SOLVER_NPN && c->solver != FEN_SOLVER_NNN) return false;
    for (int ax = 0; ax < 3; ax++) {
        const bool per = c->periodic[ax] != 0;
        for (int f : {FEN_U, FEN_V, FEN_W, FEN_P, FEN_PHI})
            for (int side = 0; side < 2; side++) {
                const int t = c->bc_type[f][2 * ax + side];
                if (per ? t != 0 : (t != 1 && t != 2)) return false;
            }
    }
    return true;
}

// How the fused kernel cuts a grid: tiles of TX x 8 cells, two rows per
// thread, marched over kb planes.
//
// Tiles are 128 wide on large grids (every tile row a 1 KB run of FP64) and
// 64 wide on small ones.  In FP64 a 128 x 8 tile's ring fills a CU (125 KB of
// LDS), a 64 x 8 one leaves room for a second workgroup whose barriers are
// its own: while the fields stay in the Infinity Cache that second workgroup
// hides more latency (128 x 128 x 160 nnn: 58 us against 64; 128 x 256 x 101
// npn: 73 against 80), and once HBM bounds the march the long rows win
// (256 x 256 x 64: 102 us against 100, 256 x 256 x 100: 172 against 182,
// 256^3: 420 against 470, 512 x 256 x 192: 635 against 746).  FP32 tiles of
// either width share a CU, and the wide ones are no slower from nx = 128
// (256^3: 235 us against 256).  (Launches back to back; inside a run, after the
// solve's passes, 128 x 128 x 160 takes 69 us, 128 x 256 x 101 87, 256^3 430 to
// 440, 512 x 256 x 192 655 and FP32 256^3 238 to 250.)
struct MarchPlan {
    bool wide;
    int nbx, nby, kb;
};

constexpr int kPMRows = 8, kPMNJ = 2;
constexpr size_t kPMWideCells = (size_t)5 << 20;

// Planes per march: a workgroup forms two planes before its first, so a cut
// into nz/kb marches costs (kb + 2) planes per march on the CU that gets most
// of them: w = ceil(workgroups / CUs), run `share` at a time.  A workgroup
// that has a CU to itself takes 0.65 of the time of two side by side (fitted at
// 128 x 256 x 101; over 54 other grids and forms of 0.8 to 5 M cells, all
// solvers, its step is within 2.6 % in FP64 and 4.8 % in FP32 of the best that
// 0.5, 0.65, 0.8 and 1 give, where 0.5 loses up to 19 % and 0.8 up to 9 %).  (At 128
// x 256 x 101 the cut that fills the chip once, kb = 13, takes 73 us, its
// neighbours 9 and 17 97 and 88 us; 512 x 256 x 192: 635 us at kb = 96, 803
// at 64, and 975 when 128 + 64 planes left half the XCDs with the long ones.)
static int march_planes(int nz, long tiles, int num_cu, int share)
{
    int best = nz;
    double least = 0.0;
    for (int n = 1; n <= nz; n++) {
        const int kb = (nz + n - 1) / n;
        if (n > 1 && kb == (nz + n - 2) / (n - 1)) continue;   // the same cut
        const long wgs = tiles * ((nz + kb - 1) / kb), w = (wgs + num_cu - 1) / num_cu;
        const double rounds = share == 2 ? (double)(w / 2) + 0.65 * (double)(w % 2) : (double)w;
        const double cost = rounds * (kb + 2);
        if (n == 1 || cost < least) {
            least = cost;
            best = kb;
        }
        if (wgs > 16L * num_cu) break;   // shorter marches only add planes
    }
    return best;
}

template <class R> static MarchPlan march_plan(const fen_ctx *c)
{
    constexpr bool f64 = std::is_same<R, double>::value;
    const Box &b = c->box;
    MarchPlan p;
    p.wide = b.nx >= 128 && (!f64 || c->n_int >= kPMWideCells);
    p.nbx = (b.nx + (p.wide ? 127 : 63)) / (p.wide ? 128 : 64);
    p.nby = (b.ny + kPMRows - 1) / kPMRows;
    p.kb = march_planes(b.nz, (long)p.nbx * p.nby, c->num_cu, f64 && p.wide ? 1 : 2);
    return p;
}

template <class R, int P2> static void launch_pm(fen_ctx *c, const PMArgs<R> &a, const MarchPlan &p, int zw, bool save)
{
    const int nbz = (c->box.nz + a.kb - 1) / a.kb;
    const dim3 grid((unsigned)((long)p.nbx * p.nby * nbz));
#define FEN_PM_TX(SRC, ZW, TX, SAVE)                                                                        \
    hipLaunchKernelGGL((project_momentum_kernel<R, SRC, ZW, kPMRows, 1, TX, SAVE, kPMNJ, P2>), grid,         \
                       dim3(TX * kPMRows / kPMNJ), 0, c->stream, a)
#define FEN_PM(SRC, ZW, SAVE)                       \
    do {                                            \
        if (p.wide) FEN_PM_TX(SRC, ZW, 128, SAVE);  \
        else FEN_PM_TX(SRC, ZW, 64, SAVE);          \
    } while (0)
    if constexpr (std::is_same<R, double>::value) {
        if (save) {
            FEN_PM(0, 0, 1);
            return;
        }
        if (zw == 2) {
            if (c->has_source) FEN_PM(1, 2, 0);
            else FEN_PM(0, 2, 0);
            return;
        }
    }
    if (zw == 1) {
        if (c->has_source) FEN_PM(1, 1, 0);
        else FEN_PM(0, 1, 0);
    } else {
        if (c->has_source) FEN_PM(1, 0, 0);
        else FEN_PM(0, 0, 0);
    }
#undef FEN_PM
#undef FEN_PM_TX
}

// Step n's projection fused with step n+1's momentum (a grid periodic in
// every direction, x, y periodic with z walls, or the general walls of
// fused_general_walls).  Step n's checks are not formed: step n+1 ends
// pending, so its own checks are what a reader asks for.
// us_in/p_in: u*, v*, w* and p of step n;
// us_out/p_out: u*, v*, w* of step n+1 and p after step n (distinct arrays);
// save (FP64, periodic grid, no source), if given: u, v, w of step n with
// their periodic images.
template <class R>
void launch_project_momentum(fen_ctx *c, double dt_p, double dt_m, double A, double B, void *const *us_in,
                             const void *p_in, void *const *us_out, void *p_out, void *const *save)
{
    const bool periodic = c->img_vel == 7 && c->img_p == 7 && c->img_phi == 7 && !c->shift_active;
    const bool zwalls = fused_z_walls(c);
    const bool general = !periodic && !zwalls && std::is_same<R, double>::value && fused_general_walls(c) &&
                         !c->shift_active;
    if (c->box.dim != 3 || !(periodic || zwalls || general))
        throw std::runtime_error("fused projection + momentum needs a periodic grid, x, y periodic with z walls, "
                                 "or the npn/nnn walls");
    PMArgs<R> a{};
    if (general) {
        a.wall = (c->periodic[0] ? 0 : 1) | (c->periodic[1] ? 0 : 2) | (c->periodic[2] ? 0 : 4);
        // packed per field: face f's bc type in bits 2f..2f+1, location in bits 12..13
        const int fid[4] = {FEN_U, FEN_V, FEN_W, FEN_P};
        const int loc[4] = {1, 2, 3, 0};
        for (int q = 0; q < 4; q++) {
            a.gtype[q] = loc[q] << 12;
            for (int f = 0; f < 6; f++) a.gtype[q] |= c->bc_type[fid[q]][f] << (2 * f);
        }
        a.gplane = reinterpret_cast<const R *const *>(c->d_plane_tab);
        if (!c->d_wallbuf) FEN_HIP_CHECK(hipMalloc(&c->d_wallbuf, 4 * pm_wall_layout(c->box).per_field * sizeof(R)));
        a.wbuf = as<R>(c->d_wallbuf);
    }
    if (zwalls) {
        a.shift = c->shift_active ? c->d_shift : nullptr;
        for (int d = 0; d < 3; d++) {
            a.zlo[d] = as<R>(c->d_plane[FEN_U + d][FEN_FRONT]);
            a.zhi[d] = as<R>(c->d_plane[FEN_U + d][FEN_BACK]);
        }
    }
    a.m = momentum_args<R>(c, dt_m, A, B);
    a.m.us = as<R>(us_out[0]); a.m.vs = as<R>(us_out[1]); a.m.ws = as<R>(us_out[2]);
    a.us = as<R>(us_in[0]); a.vs = as<R>(us_in[1]); a.ws = as<R>(us_in[2]);
    a.phi = as<R>(c->d_phi);
    a.p_in = static_cast<const R *>(p_in);
    a.p_out = as<R>(p_out);
    a.pid = 1.0 / c->delta;
    a.pdt = dt_p;
    a.prhof = 0.5 * (c->density + c->density);
    a.prpow2 = pow2_value(a.prhof) ? 1 : 0;
    a.pirhof = a.prpow2 ? 1.0 / a.prhof : 0.0;
    // how the grid is cut into tiles and marches
    const MarchPlan plan = march_plan<R>(c);
    a.m.nbx = plan.nbx;
    a.m.nby = plan.nby;
    a.kb = plan.kb;
    if (general) {
        // the state at the wall positions, read by the march below
        const long nw = pm_wall_layout(c->box).per_field;
        hipLaunchKernelGGL(wall_state_kernel<R>, dim3((unsigned)((nw + 255) / 256), 4), dim3(256), 0, c->stream, a);
    }
    if (save) {
        if (!std::is_same<R, double>::value) throw std::runtime_error("state saving is FP64");
        if (!periodic || c->has_source) throw std::runtime_error("state saving needs a periodic grid and no source");
        for (int d = 0; d < 3; d++) a.save[d] = as<R>(save[d]);
    }
    prof_begin(c, K_PROJ_MOM);
    const int zw = zwalls ? 1 : (general ? 2 : 0);
    if (a.prpow2) launch_pm<R, 1>(c, a, plan, zw, save != nullptr);
    else launch_pm<R, 0>(c, a, plan, zw, save != nullptr);
    // reads u*, v*, w*, p, phi, dv_o (+ S); writes p, u*, v*, w*, dv_o
    prof_end(c, K_PROJ_MOM, (c->has_source ? 18.0 : 15.0) * sizeof(R) * c->n_int);
}

template void launch_project_momentum<double>(fen_ctx *, double, double, double, double, void *const *, const void *,
                                              void *const *, void *, void *const *);
template void launch_project_momentum<float>(fen_ctx *, double, double, double, double, void *const *, const void *,
                                             void *const *, void *, void *const *);

}  // namespace fen
