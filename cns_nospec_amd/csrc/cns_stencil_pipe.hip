// cns_stencil_pipe.hip -- pipelined z-marching hypterm and diffterm for gfx950.
//
// The stencils of the per-kernel calls and of the unfused step (the fused step's are in
// cns_stage.hip).  A workgroup owns a TX x 8 column tile (TX = 64: 512 threads, one wave per
// row; the default is TX = 32: 256 threads, two rows per wave, two workgroups per CU) and
// marches up a run of planes.  Every field whose x/y neighbours a plane needs
// is staged in LDS as a full 16 x (TX+8) tile (4 cells of halo on each side), loaded with
// direct-to-LDS DMA (global_load_lds_dwordx4: each lane moves 16 bytes straight
// into the tile, no registers involved) into one of two LDS buffers.  The loads of
// plane k+1 are issued right after the last barrier of plane k, so that its
// compute hides their latency; a plane costs one barrier (hypterm) or
// two (diffterm), and there is no per-plane gather loop.  z neighbours of the
// lane's own column come from 9-plane register windows whose leading values are
// prefetched one plane ahead.
//
// What bounds them: with two workgroups of four waves on a CU, each wave's own chain of LDS
// reads, FP64 arithmetic and barriers (at 256^3 diffterm moves 2.9 TB/s, hypterm 3.6).  What a wave must
// not do is wait for memory: the next plane is waited for before the stores of this one join
// the queue, diffterm's two buffers are two objects and its DMA starts behind its LDS stores
// (the compiler waits for a DMA in flight at an access that might touch what it writes), and
// taps are read one by one and once each (cns_stage_tile.h).  diffterm 258 -> 202 us at
// 200x180x160 and 554 -> 462 us at 256^3, hypterm 251 -> 221 and 585 -> 528.
//
// diffterm reads wz = d(w)/dz on the cross halo as a precomputed field (wz_kernel
// below, the reference's wz temporary of cpu/diffterm.cpp:127-151 over the ghosted
// x-y extent), so no plane needs the 8 z neighbours of halo columns.
//
// Arithmetic and its order are the reference's (cpu/hypterm.cpp:11-209,
// cpu/diffterm.cpp:22-320, cpu/advance.cpp:78-153); with -ffp-contract=off the
// results are bit-identical to the reference cpu/ path and to the other kernels.
#include <cstdlib>
#include <type_traits>

#include "cns_runs.h"
#include "cns_stage_tile.h"

namespace cns {

namespace {

struct PipeRk {
    const double *d;   // difflux (interior)
    double *out;       // result (ghosted); must not alias cons
    const double *dt;  // device dt
};

// ======================================================================= hypterm
// LDS fields (centre plane): mx, my, mz, E, p, u, v.  Register windows: mx, my, mz,
// E, w, p.  With RK the update of stage 1, cons + dt (D + F) (cpu/advance.cpp:82), takes the place of
// storing F, which stage 3 overwrites: a step of which only Unew or F is not 16-byte aligned runs it
// (cns_stencil.hip has the others).  D_rho is not read: diffterm always stores 0.0 there
// (cpu/diffterm.cpp:63-68).
enum { HMX = 0, HMY, HMZ, HE, HP, HU, HV, HNF };

template <class S, bool RK>
__global__ void __launch_bounds__(S::NT, 2)
hypterm_pipe_kernel(Geom g, const double *__restrict__ cons, const double *__restrict__ q,
                    double *__restrict__ flux, double dxi0, double dxi1, double dxi2, int kz,
                    int ntx, int nty, PipeRk rk)
{
    constexpr int TILE_ = S::TILE, PX_ = S::PX;
    __shared__ double sm[2 * HNF * TILE_];

    const int t = xcd_tile(blockIdx.x, gridDim.x);
    const int bx = t % ntx, by = (t / ntx) % nty, bz = t / (ntx * nty);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // DMA issue
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
    const double dt = RK ? rk.dt[0] : 0.0;

    // first plane's tiles in flight while the windows fill
    dma_plane_s<S, HNF>(src, (int64_t)(kbeg + NG) * pg, (lds_double *)sm, td, wave, lane);

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

    __builtin_amdgcn_s_waitcnt(0xF70);
    for (int k = kbeg; k < kend; k++) {
        const int cur = (k - kbeg) & 1;
        __syncthreads();
        if (k + 1 < kend)
            dma_plane_s<S, HNF>(src, (int64_t)(k + 1 + NG) * pg, (lds_double *)sm + (cur ^ 1) * (HNF * TILE_), td, wave, lane);

        const int64_t zo = (int64_t)(k + NG) * pg + own;
        wmx[8] = nmx; wmy[8] = nmy; wmz[8] = nmz; wE[8] = nE; ww[8] = nw; wp[8] = np;
        if (inbox && k + 1 < kend) {
            const int64_t o = zo + 5 * pg;
            nmx = c_mx[o]; nmy = c_my[o]; nmz = c_mz[o]; nE = c_E[o]; nw = q_w[o]; np = q_p[o];
        }
        const int64_t fo = iidx(g, gi - NG, gj - NG, k);
        double rkd[5], rho_c = 0.0;
        if (RK && active) {
            rho_c = cons[zo];
            rkd[IRHO] = 0.0E0;
#pragma unroll
            for (int l = 1; l < NC; l++) rkd[l] = rk.d[l * g.c + fo];
        }

        // (cells past the box are computed too, for nothing: no divergent branch around the taps)
        double F[5];
        {
            // from four rows above the own cell: every tap is a non-negative constant away
            const Taps<0> s_f(sm, (unsigned)(cur * (HNF * TILE_) + me - 4 * PX_));
            constexpr int Z = 4 * PX_;
            double hs[5], A[12];
            // fields n, a, b, E, p and v of the tile at taps +o and -o
            auto load = [&](int n, int a, int b, int v, int o) {
                A[0] = s_f[n * TILE_ + Z + o]; A[1] = s_f[n * TILE_ + Z - o];
                A[2] = s_f[a * TILE_ + Z + o]; A[3] = s_f[a * TILE_ + Z - o];
                A[4] = s_f[b * TILE_ + Z + o]; A[5] = s_f[b * TILE_ + Z - o];
                A[6] = s_f[HE * TILE_ + Z + o]; A[7] = s_f[HE * TILE_ + Z - o];
                A[8] = s_f[HP * TILE_ + Z + o]; A[9] = s_f[HP * TILE_ + Z - o];
                A[10] = s_f[v * TILE_ + Z + o]; A[11] = s_f[v * TILE_ + Z - o];
            };
#define XY(FIRST, C) \
    hyp_tap<FIRST>(C, A[0], A[1], A[2], A[3], A[4], A[5], A[6], A[7], A[8], A[9], A[8], A[9], A[10], A[11], hs)
#define ZT(FIRST, C, m)                                                                                        \
    hyp_tap<FIRST>(C, wmz[4 + m], wmz[4 - m], wmx[4 + m], wmx[4 - m], wmy[4 + m], wmy[4 - m], wE[4 + m],       \
                   wE[4 - m], wp[4 + m], wp[4 - m], wp[4 + m], wp[4 - m], ww[4 + m], ww[4 - m], hs)
            load(HMX, HMY, HMZ, HU, 1);
            XY(true, ALP);
            load(HMX, HMY, HMZ, HU, 2);
            XY(false, BET);
            load(HMX, HMY, HMZ, HU, 3);
            XY(false, GAM);
            load(HMX, HMY, HMZ, HU, 4);
            XY(false, DEL);
            F[IRHO] = -(hs[0]) * dxi0;
            F[IMX] = -(hs[1]) * dxi0;
            F[IMY] = -(hs[2]) * dxi0;
            F[IMZ] = -(hs[3]) * dxi0;
            F[IENE] = -(hs[4]) * dxi0;
            load(HMY, HMX, HMZ, HV, PX_);
            XY(true, ALP);
            load(HMY, HMX, HMZ, HV, 2 * PX_);
            XY(false, BET);
            load(HMY, HMX, HMZ, HV, 3 * PX_);
            XY(false, GAM);
            load(HMY, HMX, HMZ, HV, 4 * PX_);
            XY(false, DEL);
            F[IRHO] = F[IRHO] - hs[0] * dxi1;
            F[IMY] = F[IMY] - hs[1] * dxi1;
            F[IMX] = F[IMX] - hs[2] * dxi1;
            F[IMZ] = F[IMZ] - hs[3] * dxi1;
            F[IENE] = F[IENE] - hs[4] * dxi1;
            ZT(true, ALP, 1);
            ZT(false, BET, 2);
            ZT(false, GAM, 3);
            ZT(false, DEL, 4);
            F[IRHO] = F[IRHO] - hs[0] * dxi2;
            F[IMZ] = F[IMZ] - hs[1] * dxi2;
            F[IMX] = F[IMX] - hs[2] * dxi2;
            F[IMY] = F[IMY] - hs[3] * dxi2;
            F[IENE] = F[IENE] - hs[4] * dxi2;
            pin(F[0], F[1], F[2], F[3], F[4]);
#undef XY
#undef ZT
        }
        // The next plane has landed before the stores join the queue: the barrier that opens it
        // need not wait for them.
        __builtin_amdgcn_s_waitcnt(0xF70);
        if (active) {
            const double uc[5] = {rho_c, wmx[4], wmy[4], wmz[4], wE[4]};
#pragma unroll
            for (int l = 0; l < NC; l++) {
                if (RK)
                    rk.out[l * cg + zo] = uc[l] + dt * (rkd[l] + F[l]);
                else
                    flux[l * g.c + fo] = F[l];
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
    // two objects: reads of the one then need not wait for the DMA into the other
    __shared__ __align__(16) double sm0[DNF * S::TILE], sm1[DNF * S::TILE];
    __shared__ double s_ux[S::R * S::TX];   // row r (0..15), column 4+c
    __shared__ double s_vy[S::BY * S::PX];  // row 4+r (r 0..7), column c (0..PX-1)

    const int t = xcd_tile(blockIdx.x, gridDim.x);
    const int bx = t % ntx, by = (t / ntx) % nty, bz = t / (ntx * nty);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // DMA issue
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

    dma_plane_s<S, DNF>(src, (int64_t)(kbeg + NG) * pg, (lds_double *)sm0, td, wave, lane);

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
        double a[9] = {}, b[9] = {};  // all loads of a plane at once
        if (need_ux) {
#pragma unroll
            for (int i = 0; i < 9; i++)
                if (i != 4) a[i] = q_u[o + i - 4];
        }
        if (need_vy) {
#pragma unroll
            for (int i = 0; i < 9; i++)
                if (i != 4) b[i] = q_v[o + (int64_t)(i - 4) * xg];
        }
        FENCE();
#define GUX(mm) a[4 + (mm)]
#define GVY(mm) b[4 + (mm)]
        const double ux_ = D1(GUX) * dxi0, vy_ = D1(GVY) * dxi1;
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

    auto plane = [&](int k, auto odd) {
        const double *const b = decltype(odd)::value ? sm1 : sm0;
        lds_double *const next = decltype(odd)::value ? (lds_double *)sm0 : (lds_double *)sm1;
        __syncthreads();
        ww[8] = nw;
        wt[8] = nt;
        constexpr int T = S::TILE, P = S::PX, Z = 4 * P;
        // ---------------- phase B
        {
            double a[9];
#define GA(mm) a[4 + (mm)]
            // leading plane: ux, vy of the own column (cpu/diffterm.cpp:77-81, :110-114)
            const Taps<0> p_l(b, (unsigned)(me - Z));
            wu[8] = p_l[DLU * T + Z];
            wv[8] = p_l[DLV * T + Z];
#pragma unroll
            for (int m = 0; m < 9; m++)
                if (m != 4) a[m] = p_l[DLU * T + Z + m - 4];
            wux[8] = D1(GA) * dxi0;
#pragma unroll
            for (int m = 0; m < 9; m++)
                if (m != 4) a[m] = p_l[DLV * T + m * P];
            wvy[8] = D1(GA) * dxi1;
            // centre plane, ux: the own rows from the window (ux of plane k, computed from
            // the same values four planes ago), the halo rows 0..3 and 12..15 from the tile
            s_ux[me64] = wux[4];
            {
                const int rr = threadIdx.x / S::TX, r = rr < 4 ? rr : rr + S::BY, c = threadIdx.x % S::TX;
                const Taps<0> p_u(b, (unsigned)(DCU * T + r * P + c));
#pragma unroll
                for (int m = 0; m < 9; m++)
                    if (m != 4) a[m] = p_u[m];
                s_ux[r * S::TX + c] = D1(GA) * dxi0;
            }
            // centre plane, vy: the own cells from the window, the x-halo columns 0..3 and
            // 68..71 of rows 4..11 from the tile
            s_vy[meby] = wvy[4];
            if (threadIdx.x < 8 * S::BY) {
                const int rr = threadIdx.x >> 3, cc = threadIdx.x & 7, c = cc < 4 ? cc : cc + S::TX;
                const Taps<0> p_v(b, (unsigned)(DCV * T + rr * P + c));
#pragma unroll
                for (int m = 0; m < 9; m++)
                    if (m != 4) a[m] = p_v[m * P];
                s_vy[rr * P + c] = D1(GA) * dxi1;
            }
#undef GA
        }
        __syncthreads();
        // (in flight during phase B the next plane's loads would be waited for at its LDS stores)
        if (k + 1 < kend) {
            dma_plane_s<S, DNF>(src, (int64_t)(k + 1 + NG) * pg, next, td, wave, lane);
            if (inbox) {
                const int64_t o = (int64_t)(k + NG + 5) * pg + own;
                nw = q_w[o];
                nt = q_t[o];
            }
        }

        // ---------------- phase C: z terms from the windows, x and y terms from the tiles, one
        // tap pair of all of them at a time, then the reference's sums (cpu/diffterm.cpp:159-311)
        double xu, xv, xw, xt, d2v, d2w, m1, m2, A[12];
        double uzz = CENTER * wu[4], vzz = CENTER * wv[4], wzz = CENTER * ww[4], tzz = CENTER * wt[4], uz, vz, uxz, vyz;
#define ZT(FIRST, C1, C2, m)                          \
    tap<false>(uzz, C2 * (wu[4 + m] + wu[4 - m]));    \
    tap<false>(vzz, C2 * (wv[4 + m] + wv[4 - m]));    \
    tap<false>(wzz, C2 * (ww[4 + m] + ww[4 - m]));    \
    tap<false>(tzz, C2 * (wt[4 + m] + wt[4 - m]));    \
    tap<FIRST>(uz, C1 * (wu[4 + m] - wu[4 - m]));     \
    tap<FIRST>(vz, C1 * (wv[4 + m] - wv[4 - m]));     \
    tap<FIRST>(uxz, C1 * (wux[4 + m] - wux[4 - m]));  \
    tap<FIRST>(vyz, C1 * (wvy[4 + m] - wvy[4 - m]))
        ZT(true, ALP, OFF1, 1);
        ZT(false, BET, OFF2, 2);
        ZT(false, GAM, OFF3, 3);
        ZT(false, DEL, OFF4, 4);
#undef ZT
        uzz = uzz * dxi2s;
        vzz = vzz * dxi2s;
        wzz = wzz * dxi2s;
        tzz = tzz * dxi2s;
        uz = uz * dxi2;
        vz = vz * dxi2;
        const Taps<0> s_d(b, (unsigned)(me - Z));
        // u, v, w, T, wz of the tile at taps +o and -o, vy (x) or ux (y) in the last pair
        auto load = [&](int o) {
            A[0] = s_d[DCU * T + Z + o]; A[1] = s_d[DCU * T + Z - o];
            A[2] = s_d[DCV * T + Z + o]; A[3] = s_d[DCV * T + Z - o];
            A[4] = s_d[DCW * T + Z + o]; A[5] = s_d[DCW * T + Z - o];
            A[6] = s_d[DCT * T + Z + o]; A[7] = s_d[DCT * T + Z - o];
            A[8] = s_d[DWZ * T + Z + o]; A[9] = s_d[DWZ * T + Z - o];
        };
        // second differences of u, v, w, T; first of A[2 f] (d2v), w (d2w) and of the two mixed terms
#define XY(FIRST, C1, C2, f)                         \
    tap<false>(xu, C2 * (A[0] + A[1]));              \
    tap<false>(xv, C2 * (A[2] + A[3]));              \
    tap<false>(xw, C2 * (A[4] + A[5]));              \
    tap<false>(xt, C2 * (A[6] + A[7]));              \
    tap<FIRST>(d2v, C1 * (A[2 * f] - A[2 * f + 1])); \
    tap<FIRST>(d2w, C1 * (A[4] - A[5]));             \
    tap<FIRST>(m1, C1 * (A[10] - A[11]));            \
    tap<FIRST>(m2, C1 * (A[8] - A[9]))
#define XT(FIRST, C1, C2, m)                                  \
    load(m);                                                  \
    A[10] = s_m[4 + m]; A[11] = s_m[4 - m];                   \
    XY(FIRST, C1, C2, 1)
#define YT(FIRST, C1, C2, m)                                  \
    load(m * P);                                              \
    A[10] = s_n[(4 + m) * S::TX]; A[11] = s_n[(4 - m) * S::TX]; \
    XY(FIRST, C1, C2, 0)
        const Taps<0> s_m(s_vy, (unsigned)(meby - 4)), s_n(s_ux, (unsigned)(me64 - 4 * S::TX));
        xu = CENTER * wu[4]; xv = CENTER * wv[4]; xw = CENTER * ww[4]; xt = CENTER * wt[4];
        XT(true, ALP, OFF1, 1);
        XT(false, BET, OFF2, 2);
        XT(false, GAM, OFF3, 3);
        XT(false, DEL, OFF4, 4);
        const double uxx = xu * dxi0s, vxx = xv * dxi0s, wxx = xw * dxi0s, txx = xt * dxi0s;
        const double vx = d2v * dxi0, wx = d2w * dxi0, vyx = m1 * dxi0, wzx = m2 * dxi0;
        xu = CENTER * wu[4]; xv = CENTER * wv[4]; xw = CENTER * ww[4]; xt = CENTER * wt[4];
        YT(true, ALP, OFF1, 1);
        YT(false, BET, OFF2, 2);
        YT(false, GAM, OFF3, 3);
        YT(false, DEL, OFF4, 4);
#undef XY
#undef XT
#undef YT
        const double uyy = xu * dxi1s, vyy = xv * dxi1s, wyy = xw * dxi1s, tyy = xt * dxi1s;
        const double uy = d2v * dxi1, wy = d2w * dxi1, uxy = m1 * dxi1, wzy = m2 * dxi1;
        uxz = uxz * dxi2;
        vyz = vyz * dxi2;
        const double dmx = eta * (FourThirds * uxx + uyy + uzz + OneThird * (vyx + wzx));
        const double dmy = eta * (vxx + FourThirds * vyy + vzz + OneThird * (uxy + wzy));
        const double dmz = eta * (wxx + wyy + FourThirds * wzz + OneThird * (uxz + vyz));
        const double ux = wux[4], vy = wvy[4], wz = s_d[DWZ * T + Z];
        const double divu = TwoThirds * (ux + vy + wz);
        const double tauxx = 2.E0 * ux - divu;
        const double tauyy = 2.E0 * vy - divu;
        const double tauzz = 2.E0 * wz - divu;
        const double tauxy = uy + vx;
        const double tauxz = uz + wx;
        const double tauyz = vz + wy;
        double mechwork = tauxx * ux + tauyy * vy + tauzz * wz + (tauxy * tauxy) + (tauxz * tauxz) + (tauyz * tauyz);
        mechwork = eta * mechwork + dmx * wu[4] + dmy * wv[4] + dmz * ww[4];
        double dE = alam * (txx + tyy + tzz) + mechwork;
        pin(dE);
        // The next plane has landed before the stores join the queue: the barrier that opens it
        // need not wait for them.
        __builtin_amdgcn_s_waitcnt(0xF70);
        if (active) {
            const int64_t fo = iidx(g, gi - NG, gj - NG, k);
            const int64_t c = g.c;
            difflux[fo] = 0.0E0;
            difflux[fo + IMX * c] = dmx;
            difflux[fo + IMY * c] = dmy;
            difflux[fo + IMZ * c] = dmz;
            difflux[fo + IENE * c] = dE;
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
    };
    __builtin_amdgcn_s_waitcnt(0xF70);
#pragma unroll 1
    for (int k = kbeg; k < kend; k += 2) {
        plane(k, std::false_type());
        if (k + 1 < kend) plane(k + 1, std::true_type());
    }
}

// z runs.  A launch takes ceil(workgroups / slots) rounds of (planes + the window fill, which
// costs `warm` planes: its prologue differences u and v of eight planes for diffterm, 3,
// and only loads for hypterm, 1); the run length that makes this smallest is taken, and of
// runs within 1 % the shortest, which start their neighbours' planes closer in time.  Halving
// until 2048 workgroups, as before, left a last round nearly empty or the runs at twice
// the fill: diffterm 324 -> 272 us at 200x180x160, 76 -> 54 us at 130x97x61, 712 -> 655 us at
// 256^3; hypterm 58 -> 39 us at 130x97x61 (all before the planes stopped waiting for memory).
// CNS_PIPE_KZ in the environment caps the run length (for measurements).
int pipe_kz(const Geom &g, int64_t tiles, int slots, int warm)
{
    static const int cap = [] {
        const char *e = getenv("CNS_PIPE_KZ");
        return e ? atoi(e) : 0;
    }();
    return pipe_run(g.n2, cap >= 4 && cap < g.n2 ? cap : g.n2, tiles, slots, warm);
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
                                 double dxi1, double dxi2, const PipeRk &rk, hipStream_t s)
{
    const int ntx = (g.n0 + S::TX - 1) / S::TX, nty = (g.n1 + S::BY - 1) / S::BY;
    const int kz = pipe_kz(g, (int64_t)ntx * nty, S::TX == 32 ? 512 : 256, 1);
    const int nb = ntx * nty * ((g.n2 + kz - 1) / kz);
    if (rk.out)
        hypterm_pipe_kernel<S, true><<<nb, S::NT, 0, s>>>(g, cons, q, flux, dxi0, dxi1, dxi2, kz, ntx, nty, rk);
    else
        hypterm_pipe_kernel<S, false><<<nb, S::NT, 0, s>>>(g, cons, q, flux, dxi0, dxi1, dxi2, kz, ntx, nty, rk);
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

static hipError_t launch_hyp_pipe(const Geom &g, const double *cons, const double *q, double *flux, const double dxi[3],
                                  const PipeRk &rk, hipStream_t s)
{
    if (wide_tiles("CNS_HYP_TX"))
        return launch_hyp_pipe_shape<Shape<64>>(g, cons, q, flux, dxi[0], dxi[1], dxi[2], rk, s);
    return launch_hyp_pipe_shape<Shape<32>>(g, cons, q, flux, dxi[0], dxi[1], dxi[2], rk, s);
}

hipError_t launch_hypterm_pipe(const Geom &g, const double *cons, const double *q, double *flux, const double dxi[3],
                               hipStream_t s)
{
    return launch_hyp_pipe(g, cons, q, flux, dxi, PipeRk{}, s);
}

hipError_t launch_hypterm_pipe_rk1(const Geom &g, const double *cons, const double *q, const double dxi[3],
                                   const double *d, double *out, const double *dt_dev, hipStream_t s)
{
    return launch_hyp_pipe(g, cons, q, nullptr, dxi, PipeRk{d, out, dt_dev}, s);
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
