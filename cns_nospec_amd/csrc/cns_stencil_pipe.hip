// cns_stencil_pipe.hip -- pipelined z-marching hypterm and diffterm for gfx950.
//
// The stencils of the per-kernel calls and of the unfused step (the fused step's are in
// cns_stage.hip).  A workgroup owns a TX x 8 column tile (TX = 64: 512 threads, one wave per
// row; the default is TX = 32: 256 threads, two rows per wave, two workgroups per CU) and
// marches up a run of planes.  Every field whose x/y neighbours a plane needs
// is staged in LDS as a full 16 x (TX+8) tile (4 cells of halo on each side), loaded with
// direct-to-LDS DMA (global_load_lds_dwordx4: each lane moves 16 bytes straight
// into the tile, no registers involved) into one of two LDS buffers.  The loads of
// plane k+1 are issued right after the barrier that opens plane k, so the whole
// compute of plane k hides their latency; a plane costs one barrier (hypterm) or
// two (diffterm), and there is no per-plane gather loop.  z neighbours of the
// lane's own column come from 9-plane register windows whose leading values are
// prefetched one plane ahead.
//
// diffterm reads wz = d(w)/dz on the cross halo as a precomputed field (wz_kernel
// below, the reference's wz temporary of cpu/diffterm.cpp:127-151 over the ghosted
// x-y extent), so no plane needs the 8 z neighbours of halo columns.
//
// Arithmetic and its order are the reference's (cpu/hypterm.cpp:11-209,
// cpu/diffterm.cpp:22-320, cpu/advance.cpp:78-153); with -ffp-contract=off the
// results are bit-identical to the reference cpu/ path and to the other kernels.
#include <cstdlib>

#include "cns_pipe_tile.h"

namespace cns {

namespace {

struct PipeRk {
    const double *d;     // difflux (interior)
    const double *base;  // U^n (ghosted), phases 2 and 3
    double *out;         // result (ghosted); must not alias cons
    const double *dt;    // device dt
    int phase;           // 0: plain hypterm
};

// ======================================================================= hypterm
// LDS fields (centre plane): mx, my, mz, E, p, u, v.  Register windows: mx, my, mz,
// E, w, p.  With RK the stage update of the cell is applied as in cns_stencil.hip,
// with three savings of HBM traffic that leave every result bit-identical:
//  * D_rho is not read: diffterm always stores 0.0 there (cpu/diffterm.cpp:63-68);
//  * STAGE1: the base is cons itself, so the update is cons + dt*(D+F), the
//    reference's own form (cpu/advance.cpp:82), without re-reading the base;
//  * !WRITE_F: flux is not stored (stages 1 and 2 of a step, whose F the third
//    stage overwrites).
enum { HMX = 0, HMY, HMZ, HE, HP, HU, HV, HNF };

template <class S, bool RK, bool STAGE1, bool WRITE_F>
__global__ void __launch_bounds__(S::NT, 2)
hypterm_pipe_kernel(Geom g, const double *__restrict__ cons, const double *__restrict__ q,
                    double *__restrict__ flux, double dxi0, double dxi1, double dxi2, int kz,
                    int ntx, int nty, PipeRk rk)
{
    constexpr int TILE_ = S::TILE, PX_ = S::PX;
    __shared__ double sm[2 * HNF * TILE_];

    const int t = xcd_tile(blockIdx.x, gridDim.x);
    const int bx = t % ntx, by = (t / ntx) % nty, bz = t / (ntx * nty);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;       // DMA issue
    const int col = threadIdx.x % S::TX, row = threadIdx.x / S::TX;  // the lane's cell
    const TileDma td{bx * S::TX, by * S::BY, g.g1 - 1, g.xg - 2, (unsigned)g.xg};
    const int gi = td.gi0 + col + 4, gj = td.gj0 + row + 4;
    const bool inbox = gi < g.g0 && gj < g.g1;
    const bool active = gi < g.n0 + NG && gj < g.n1 + NG;
    const int kbeg = bz * kz, kend = min(kbeg + kz, g.n2);
    const int64_t cg = g.cg, pg = g.pg;
    const double *c_mx = cons + IMX * cg, *c_my = cons + IMY * cg, *c_mz = cons + IMZ * cg,
                 *c_E = cons + IENE * cg;
    const double *q_u = q + QU * cg, *q_v = q + QV * cg, *q_w = q + QW * cg, *q_p = q + QPRES * cg;
    const double *const src[HNF] = {c_mx, c_my, c_mz, c_E, q_p, q_u, q_v};
    const int64_t own = (int64_t)gj * g.xg + gi;
    const int me = (row + 4) * PX_ + col + 4;
    double dt = 0.0, ra = 0.0, rb = 1.0;
    if (RK) {
        // r = ra*base + rb*(cons + dt*(D+F)) with (ra, rb) = (0, 1), (3/4, 1/4), (1/3, 2/3):
        // 0*base + 1*x is exactly x, so each phase keeps the reference's rounding
        // (cpu/advance.cpp:82, :114-116, :148-150)
        dt = rk.dt[0];
        ra = rk.phase == 1 ? 0.0E0 : (rk.phase == 2 ? ThreeQuarters : OneThird);
        rb = rk.phase == 1 ? 1.0E0 : (rk.phase == 2 ? OneQuarter : TwoThirds);
    }

    // first plane's tiles in flight while the windows fill
    dma_plane_s<S, HNF>(src, (int64_t)(kbeg + NG) * pg, sm, td, wave, lane);

    double wmx[9], wmy[9], wmz[9], wE[9], ww[9], wp[9];
    double nmx = 0, nmy = 0, nmz = 0, nE = 0, nw = 0, np = 0;
    if (inbox) {
#pragma unroll
        for (int m = 0; m < 8; m++) {
            const int64_t o = (int64_t)(kbeg + m) * pg + own;
            wmx[m] = c_mx[o]; wmy[m] = c_my[o]; wmz[m] = c_mz[o];
            wE[m] = c_E[o]; ww[m] = q_w[o]; wp[m] = q_p[o];
        }
        const int64_t o = (int64_t)(kbeg + 2 * NG) * pg + own;
        nmx = c_mx[o]; nmy = c_my[o]; nmz = c_mz[o]; nE = c_E[o]; nw = q_w[o]; np = q_p[o];
    }

    for (int k = kbeg; k < kend; k++) {
        const int cur = (k - kbeg) & 1;
        const double *b = sm + cur * (HNF * TILE_);
        plane_barrier();
        if (k + 1 < kend)
            dma_plane_s<S, HNF>(src, (int64_t)(k + 1 + NG) * pg, sm + (cur ^ 1) * (HNF * TILE_), td, wave, lane);

        const int64_t zo = (int64_t)(k + NG) * pg + own;
        wmx[8] = nmx; wmy[8] = nmy; wmz[8] = nmz; wE[8] = nE; ww[8] = nw; wp[8] = np;
        if (inbox && k + 1 < kend) {
            const int64_t o = zo + 5 * pg;
            nmx = c_mx[o]; nmy = c_my[o]; nmz = c_mz[o]; nE = c_E[o]; nw = q_w[o]; np = q_p[o];
        }
        const int64_t fo = iidx(g, gi - NG, gj - NG, k);
        double rkd[5], rkb[5], rho_c = 0.0;
        if (RK && active) {
            rho_c = cons[zo];
            rkd[IRHO] = 0.0E0;
#pragma unroll
            for (int l = 0; l < NC; l++) {
                if (l != IRHO) rkd[l] = rk.d[l * g.c + fo];
                if (!STAGE1) rkb[l] = rk.base[l * cg + zo];
            }
        }

        if (active) {
            const double *s_mx = b + HMX * TILE_, *s_my = b + HMY * TILE_, *s_mz = b + HMZ * TILE_,
                         *s_E = b + HE * TILE_, *s_p = b + HP * TILE_, *s_u = b + HU * TILE_,
                         *s_v = b + HV * TILE_;
            double F[5];
            hyp_flux<PX_>(s_mx, s_my, s_mz, s_E, s_p, s_u, s_v, me, wmx, wmy, wmz, wE, ww, wp, dxi0, dxi1, dxi2, F);
            if (RK) {
                const double uc[5] = {rho_c, wmx[4], wmy[4], wmz[4], wE[4]};
                double o[5];
                rk_store<STAGE1, WRITE_F>(F, uc, rkd, rkb, ra, rb, dt, flux, fo, g.c, rk.out, zo, cg, o);
            } else {
#pragma unroll
                for (int l = 0; l < NC; l++) flux[l * g.c + fo] = F[l];
            }
        }
#pragma unroll
        for (int m = 0; m < 8; m++) {
            wmx[m] = wmx[m + 1]; wmy[m] = wmy[m + 1]; wmz[m] = wmz[m + 1];
            wE[m] = wE[m + 1]; ww[m] = ww[m + 1]; wp[m] = wp[m + 1];
        }
    }
}

// ============================================================================ wz
// wz(i, j, k) = D1_z(w) * dxinv(3) for every (i, j) of the ghosted x-y extent and
// interior k (cpu/diffterm.cpp:126-151), into a one-component array with the ghosted
// layout (plane k+ng).  One thread per column and run of kz planes, 9-plane window.
__global__ void __launch_bounds__(256)
wz_kernel(Geom g, const double *__restrict__ q_w, double *__restrict__ wz, double dxi2, int kz)
{
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;  // j*xg + i
    if (p >= g.pg || (int)(p % g.xg) >= g.g0) return;
    const int kbeg = blockIdx.y * kz, kend = min(kbeg + kz, g.n2);
    const int64_t pg = g.pg;
    double w[9];
#pragma unroll
    for (int m = 0; m < 8; m++) w[m] = q_w[(int64_t)(kbeg + m) * pg + p];
    for (int k = kbeg; k < kend; k++) {
        w[8] = q_w[(int64_t)(k + 2 * NG) * pg + p];
#define WZ(mm) w[4 + (mm)]
        wz[(int64_t)(k + NG) * pg + p] = D1(WZ) * dxi2;
#undef WZ
#pragma unroll
        for (int m = 0; m < 8; m++) w[m] = w[m + 1];
    }
}

// ====================================================================== diffterm
// LDS fields, double-buffered: centre plane u, v (square halos), w, T, wz (cross
// halos), leading plane (k+4) u and v.  Single-buffered: ux on the tile and y-halo
// rows, vy on the tile and x-halo columns.  Per plane:
//  B  (after the opening barrier) ux, vy of the leading plane into the register
//     windows; ux, vy of the centre plane on their halos into LDS;
//  C  (after a second barrier) every output of cpu/diffterm.cpp:155-315 for the cell.
// Register windows: u, v, w, T and the computed ux, vy.
enum { DCU = 0, DCV, DCW, DCT, DWZ, DLU, DLV, DNF };

template <class S>
__global__ void __launch_bounds__(S::NT, 2)
diffterm_pipe_kernel(Geom g, const double *__restrict__ q, const double *__restrict__ wzf,
                     double *__restrict__ difflux, double dxi0, double dxi1, double dxi2, double eta,
                     double alam, int kz, int ntx, int nty)
{
    __shared__ double sm[2 * DNF * S::TILE];
    __shared__ double s_ux[S::R * S::TX];   // row r (0..15), column 4+c
    __shared__ double s_vy[S::BY * S::PX];  // row 4+r (r 0..7), column c (0..PX-1)

    const int t = xcd_tile(blockIdx.x, gridDim.x);
    const int bx = t % ntx, by = (t / ntx) % nty, bz = t / (ntx * nty);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;       // DMA issue
    const int col = threadIdx.x % S::TX, row = threadIdx.x / S::TX;  // the lane's cell
    const TileDma td{bx * S::TX, by * S::BY, g.g1 - 1, g.xg - 2, (unsigned)g.xg};
    const int gi = td.gi0 + col + 4, gj = td.gj0 + row + 4;
    const bool inbox = gi < g.g0 && gj < g.g1;
    const bool active = gi < g.n0 + NG && gj < g.n1 + NG;
    const int kbeg = bz * kz, kend = min(kbeg + kz, g.n2);
    const int64_t cg = g.cg, pg = g.pg, xg = g.xg;
    const double *q_u = q + QU * cg, *q_v = q + QV * cg, *q_w = q + QW * cg, *q_t = q + QTEMP * cg;
    const double *const src[DNF] = {q_u, q_v, q_w, q_t, wzf, q_u + 4 * pg, q_v + 4 * pg};
    const int64_t own = (int64_t)gj * xg + gi;
    const int me = (row + 4) * S::PX + col + 4;  // own cell in R x PX tiles
    const int me64 = (row + 4) * S::TX + col;    // own cell in s_ux
    const int meby = row * S::PX + col + 4;      // own cell in s_vy
    const double dxi0s = dxi0 * dxi0, dxi1s = dxi1 * dxi1, dxi2s = dxi2 * dxi2;

    dma_plane_s<S, DNF>(src, (int64_t)(kbeg + NG) * pg, sm, td, wave, lane);

    // windows: plane k+m at [4+m]; ux and vy of the first 8 planes straight from
    // global memory (the same expressions as the per-plane path)
    // The tile's own-row ux and own-cell vy feed phase B's LDS planes (uxy, vyx of the
    // neighbours), so ux is needed on every x-interior lane of the ghosted y range and
    // vy on every y-interior lane of the ghosted x range; both stencils stay in bounds.
    double wu[9], wv[9], ww[9], wt[9], wux[9], wvy[9];
    double nw = 0.0, nt = 0.0;
    const bool need_ux = gi < g.n0 + NG && gj < g.g1, need_vy = gj < g.n1 + NG && gi < g.g0;
#pragma unroll 1
    for (int m = 0; m < 8; m++) {
        const int64_t o = (int64_t)(kbeg + m) * pg + own;
        double ux_ = 0.0, vy_ = 0.0;
#define GUX(mm) q_u[o + (mm)]
#define GVY(mm) q_v[o + (int64_t)(mm) * xg]
        if (need_ux) ux_ = D1(GUX) * dxi0;
        if (need_vy) vy_ = D1(GVY) * dxi1;
#undef GUX
#undef GVY
#pragma unroll
        for (int mm = 0; mm < 7; mm++) {
            wux[mm] = wux[mm + 1];
            wvy[mm] = wvy[mm + 1];
        }
        wux[7] = ux_;
        wvy[7] = vy_;
    }
    if (inbox) {
#pragma unroll
        for (int m = 0; m < 8; m++) {
            const int64_t o = (int64_t)(kbeg + m) * pg + own;
            wu[m] = q_u[o]; wv[m] = q_v[o]; ww[m] = q_w[o]; wt[m] = q_t[o];
        }
        const int64_t o = (int64_t)(kbeg + 2 * NG) * pg + own;
        nw = q_w[o];
        nt = q_t[o];
    }

    for (int k = kbeg; k < kend; k++) {
        const int cur = (k - kbeg) & 1;
        const double *b = sm + cur * (DNF * S::TILE);
        plane_barrier();
        if (k + 1 < kend)
            dma_plane_s<S, DNF>(src, (int64_t)(k + 1 + NG) * pg, sm + (cur ^ 1) * (DNF * S::TILE), td, wave, lane);
        const double *s_cu = b + DCU * S::TILE, *s_cv = b + DCV * S::TILE, *s_cw = b + DCW * S::TILE,
                     *s_ct = b + DCT * S::TILE, *s_wz = b + DWZ * S::TILE, *s_lu = b + DLU * S::TILE,
                     *s_lv = b + DLV * S::TILE;

        const int64_t zo = (int64_t)(k + NG) * pg + own;
        wu[8] = s_lu[me];
        wv[8] = s_lv[me];
        ww[8] = nw;
        wt[8] = nt;
        if (inbox && k + 1 < kend) {
            const int64_t o = zo + 5 * pg;
            nw = q_w[o];
            nt = q_t[o];
        }

        // ---------------- phase B
        {
#define LUX(mm) s_lu[me + (mm)]
#define LVY(mm) s_lv[me + (mm) * S::PX]
            // leading plane: ux, vy of the own column (cpu/diffterm.cpp:77-81, :110-114)
            wux[8] = D1(LUX) * dxi0;
            wvy[8] = D1(LVY) * dxi1;
#undef LUX
#undef LVY
            // centre plane, ux: the own rows from the window (ux of plane k, computed from
            // the same values four planes ago), the halo rows 0..3 and 12..15 from the tile
            s_ux[me64] = wux[4];
            {
                const int rr = threadIdx.x / S::TX, r = rr < 4 ? rr : rr + S::BY, c = threadIdx.x % S::TX;
                const int l = r * S::PX + c + 4;
#define CUX(mm) s_cu[l + (mm)]
                s_ux[r * S::TX + c] = D1(CUX) * dxi0;
#undef CUX
            }
            // centre plane, vy: the own cells from the window, the x-halo columns 0..3 and
            // 68..71 of rows 4..11 from the tile
            s_vy[meby] = wvy[4];
            if (threadIdx.x < 8 * S::BY) {
                const int rr = threadIdx.x >> 3, cc = threadIdx.x & 7, c = cc < 4 ? cc : cc + S::TX;
                const int l = (rr + 4) * S::PX + c;
#define CVY(mm) s_cv[l + (mm) * S::PX]
                s_vy[rr * S::PX + c] = D1(CVY) * dxi1;
#undef CVY
            }
        }
        __syncthreads();

        // ---------------- phase C
        if (active) {
#define XS(a, mm) a[me + (mm)]
#define YS(a, mm) a[me + (mm) * S::PX]
#define CUx(mm) XS(s_cu, mm)
#define CUy(mm) YS(s_cu, mm)
#define CUz(mm) wu[4 + (mm)]
#define CVx(mm) XS(s_cv, mm)
#define CVy(mm) YS(s_cv, mm)
#define CVz(mm) wv[4 + (mm)]
#define CWx(mm) XS(s_cw, mm)
#define CWy(mm) YS(s_cw, mm)
#define CWz(mm) ww[4 + (mm)]
#define CTx(mm) XS(s_ct, mm)
#define CTy(mm) YS(s_ct, mm)
#define CTz(mm) wt[4 + (mm)]
#define VYx(mm) s_vy[meby + (mm)]
#define WZx(mm) XS(s_wz, mm)
#define UXy(mm) s_ux[me64 + (mm) * S::TX]
#define WZy(mm) YS(s_wz, mm)
#define UXz(mm) wux[4 + (mm)]
#define VYz(mm) wvy[4 + (mm)]
            // cpu/diffterm.cpp:159-187
            const double uxx = D2(CUx) * dxi0s;
            const double uyy = D2(CUy) * dxi1s;
            const double uzz = D2(CUz) * dxi2s;
            const double vyx = D1(VYx) * dxi0;
            const double wzx = D1(WZx) * dxi0;
            const double dmx = eta * (FourThirds * uxx + uyy + uzz + OneThird * (vyx + wzx));
            // :198-226
            const double vxx = D2(CVx) * dxi0s;
            const double vyy = D2(CVy) * dxi1s;
            const double vzz = D2(CVz) * dxi2s;
            const double uxy = D1(UXy) * dxi1;
            const double wzy = D1(WZy) * dxi1;
            const double dmy = eta * (vxx + FourThirds * vyy + vzz + OneThird * (uxy + wzy));
            // :237-265
            const double wxx = D2(CWx) * dxi0s;
            const double wyy = D2(CWy) * dxi1s;
            const double wzz = D2(CWz) * dxi2s;
            const double uxz = D1(UXz) * dxi2;
            const double vyz = D1(VYz) * dxi2;
            const double dmz = eta * (wxx + wyy + FourThirds * wzz + OneThird * (uxz + vyz));
            // :276-311
            const double txx = D2(CTx) * dxi0s;
            const double tyy = D2(CTy) * dxi1s;
            const double tzz = D2(CTz) * dxi2s;
            const double ux = wux[4], vy = wvy[4], wz = s_wz[me];
            const double uy = D1(CUy) * dxi1, uz = D1(CUz) * dxi2;
            const double vx = D1(CVx) * dxi0, vz = D1(CVz) * dxi2;
            const double wx = D1(CWx) * dxi0, wy = D1(CWy) * dxi1;
            const double divu = TwoThirds * (ux + vy + wz);
            const double tauxx = 2.E0 * ux - divu;
            const double tauyy = 2.E0 * vy - divu;
            const double tauzz = 2.E0 * wz - divu;
            const double tauxy = uy + vx;
            const double tauxz = uz + wx;
            const double tauyz = vz + wy;
            double mechwork = tauxx * ux + tauyy * vy + tauzz * wz + (tauxy * tauxy) + (tauxz * tauxz)
                              + (tauyz * tauyz);
            mechwork = eta * mechwork + dmx * wu[4] + dmy * wv[4] + dmz * ww[4];
            const int64_t fo = iidx(g, gi - NG, gj - NG, k);
            const int64_t c = g.c;
            difflux[fo] = 0.0E0;
            difflux[fo + IMX * c] = dmx;
            difflux[fo + IMY * c] = dmy;
            difflux[fo + IMZ * c] = dmz;
            difflux[fo + IENE * c] = alam * (txx + tyy + tzz) + mechwork;
#undef XS
#undef YS
#undef CUx
#undef CUy
#undef CUz
#undef CVx
#undef CVy
#undef CVz
#undef CWx
#undef CWy
#undef CWz
#undef CTx
#undef CTy
#undef CTz
#undef VYx
#undef WZx
#undef UXy
#undef WZy
#undef UXz
#undef VYz
        }
#pragma unroll
        for (int m = 0; m < 8; m++) {
            wu[m] = wu[m + 1];
            wv[m] = wv[m + 1];
            ww[m] = ww[m + 1];
            wt[m] = wt[m + 1];
            wux[m] = wux[m + 1];
            wvy[m] = wvy[m + 1];
        }
    }
}

// z runs.  A launch takes ceil(workgroups / slots) rounds of (planes + the window fill, which
// costs `warm` planes: its prologue differences u and v of eight planes for diffterm, 3,
// and only loads for hypterm, 1); the run length that makes this smallest is taken, and of
// runs within 1 % the shortest, which start their neighbours' planes closer in time.  Halving
// until 2048 workgroups, as before, left a last round nearly empty or the runs at twice
// the fill: diffterm 324 -> 272 us at 200x180x160, 76 -> 54 us at 130x97x61, 712 -> 655 us at
// 256^3; hypterm 58 -> 39 us at 130x97x61.
// CNS_PIPE_KZ in the environment caps the run length (for measurements).
int pipe_kz(const Geom &g, int64_t tiles, int slots, int warm)
{
    static const int cap = [] {
        const char *e = getenv("CNS_PIPE_KZ");
        return e ? atoi(e) : 0;
    }();
    const int most = cap >= 4 && cap < g.n2 ? cap : g.n2;
    int best = most;
    int64_t cost = INT64_MAX / 2;
    for (int nz = (g.n2 + most - 1) / most; nz <= g.n2; nz++) {
        const int kz = (g.n2 + nz - 1) / nz, runs = (g.n2 + kz - 1) / kz;
        const int64_t c = (tiles * runs + slots - 1) / slots * (kz + warm);
        if (c > cost + cost / 100) continue;
        best = kz;
        if (c < cost) cost = c;
    }
    return best;
}

// The stencils run on 32 x 8 tiles, two workgroups per CU (512^3: diffterm
// 4.84 -> 4.33 ms, fused hypterm 6.65 -> 6.05 ms against 64 x 8); setting the named
// variable to 64 selects 64 x 8 tiles (the results are the same bits either way).
bool wide_tiles(const char *var)
{
    const char *e = getenv(var);
    return e && atoi(e) == 64;
}

template <class S>
hipError_t launch_hyp_pipe_shape(const Geom &g, const double *cons, const double *q, double *flux, double dxi0,
                                 double dxi1, double dxi2, const double *d, const double *base, double *out,
                                 const double *dt_dev, int phase, bool write_f, hipStream_t s)
{
    const int ntx = (g.n0 + S::TX - 1) / S::TX, nty = (g.n1 + S::BY - 1) / S::BY;
    const int kz = pipe_kz(g, (int64_t)ntx * nty, S::TX == 32 ? 512 : 256, 1);
    const int nb = ntx * nty * ((g.n2 + kz - 1) / kz);
    PipeRk rk{d, base, out, dt_dev, phase};
    const bool stage1 = phase == 1 && base == cons;
#define HYP_PIPE(RK, S1, WF)                                                                              \
    hypterm_pipe_kernel<S, RK, S1, WF><<<nb, S::NT, 0, s>>>(g, cons, q, flux, dxi0, dxi1, dxi2, kz, ntx, nty, \
                                                            rk)
    if (!phase)
        HYP_PIPE(false, false, true);
    else if (stage1)
        write_f ? HYP_PIPE(true, true, true) : HYP_PIPE(true, true, false);
    else
        write_f ? HYP_PIPE(true, false, true) : HYP_PIPE(true, false, false);
#undef HYP_PIPE
    return hipGetLastError();
}

template <class S>
hipError_t launch_diffterm_shape(const Geom &g, const double *q, const double *wz, double *difflux,
                                 double dxi0, double dxi1, double dxi2, double eta, double alam,
                                 hipStream_t s)
{
    const int ntx = (g.n0 + S::TX - 1) / S::TX, nty = (g.n1 + S::BY - 1) / S::BY;
    const int kz = pipe_kz(g, (int64_t)ntx * nty, S::TX == 32 ? 512 : 256, 3);
    const int nb = ntx * nty * ((g.n2 + kz - 1) / kz);
    diffterm_pipe_kernel<S><<<nb, S::NT, 0, s>>>(g, q, wz, difflux, dxi0, dxi1, dxi2, eta, alam, kz, ntx, nty);
    return hipGetLastError();
}

}  // namespace

bool pipe_aligned(const void *p) { return ((uintptr_t)p & 15) == 0; }

hipError_t launch_hypterm_pipe(const Geom &g, const double *cons, const double *q, double *flux,
                               double dxi0, double dxi1, double dxi2, const double *d,
                               const double *base, double *out, const double *dt_dev, int phase,
                               bool write_f, hipStream_t s)
{
    if (wide_tiles("CNS_HYP_TX"))
        return launch_hyp_pipe_shape<Shape<64>>(g, cons, q, flux, dxi0, dxi1, dxi2, d, base, out, dt_dev, phase,
                                                write_f, s);
    return launch_hyp_pipe_shape<Shape<32>>(g, cons, q, flux, dxi0, dxi1, dxi2, d, base, out, dt_dev, phase,
                                            write_f, s);
}

hipError_t launch_wz(const Geom &g, const double *q, double *wz, double dxi2, hipStream_t s)
{
    const int64_t cols = (g.pg + 255) / 256;
    // runs long enough that the 8-plane window warm-up stays small; small boxes shorten them,
    // down to 8 planes, until the launch has 512 workgroups
    int kz = g.n2 > 128 ? 128 : g.n2;
    while (kz > 8 && cols * ((g.n2 + kz - 1) / kz) < 512) kz = kz / 2 > 8 ? kz / 2 : 8;
    const dim3 grid((unsigned)cols, (unsigned)((g.n2 + kz - 1) / kz));
    wz_kernel<<<grid, 256, 0, s>>>(g, q + QW * g.cg, wz, dxi2, kz);
    return hipGetLastError();
}

hipError_t launch_diffterm_pipe(const Geom &g, const double *q, const double *wz, double *difflux,
                                double dxi0, double dxi1, double dxi2, double eta, double alam,
                                hipStream_t s)
{
    if (wide_tiles("CNS_DIFF_TX"))
        return launch_diffterm_shape<Shape<64>>(g, q, wz, difflux, dxi0, dxi1, dxi2, eta, alam, s);
    return launch_diffterm_shape<Shape<32>>(g, q, wz, difflux, dxi0, dxi1, dxi2, eta, alam, s);
}

}  // namespace cns
