// cns_stage.hip -- one RK stage of the step in a single z-marching kernel (gfx950).
//
// From the ghosted conserved state alone a workgroup produces, for its 32 x 16 column tile
// and run of planes, the viscous and inviscid terms of each cell (cpu/diffterm.cpp,
// cpu/hypterm.cpp) and its SSP-RK3 update.  Primitives, their derivatives, D and F live in
// LDS and registers only: a stage reads the five conserved fields (and the stage base) and
// writes the result, where separate kernels pass Q, wz and D through memory.
//
// Storage.  512 threads, one workgroup per CU, two waves per SIMD of 256 registers each.
// Registers: 9-plane z windows of mx, my, mz, E, 1/rho, p, T and of the computed ux, vy of
// the lane's own column (u, v, w of a window plane are one product with 1/rho: ctoprim's
// own), 144 registers between planes.  LDS, 158 KB: the centre plane's raw fields as
// 24 x 40 tiles and the leading plane's own and halo cells, both loaded by direct-to-LDS
// DMA; the derived u, v, w, T, p tiles; the leading plane's u rows and v columns; an 8-plane
// ring of w on the tile's halo columns; ux, vy, wz of the centre plane with the halos
// their mixed derivatives need.
//
// Plane k (leading plane k+4):
//   1  primitives of the leading own cell into the windows, of the leading halo cells into
//      the lead tiles and the ring, of the centre plane's halo cells into the derived tiles
//      (the own cells come from the windows);
//   B
//   2  DMA of the next leading plane; ux, vy of the leading plane into the windows; ux, vy, wz
//      of the centre plane into LDS; every z term, from the windows; hypterm's x and y
//      terms, from the tiles;
//   C
//   3  DMA of the next centre plane; diffterm's x and y terms; the update and the stores;
//   A
// Before the first centre plane the windows and the ring are filled with eight planes at once.
//
// What bounds it: each wave's own chain.  A plane is 1120 to 1200 vector, 150 to 250 scalar and
// 250 LDS instructions a wave (about 1020 FP64); a wave issues an FP64 instruction every 4.2 cycles at
// best, 6.5 when it waits for the one before, two waves of a SIMD do not slow each other, and a
// plane takes 14 to 17 thousand cycles: 45 % issuing, 25 % ready and not issued, 30 % in waits
// and barriers.  More waves would need fewer registers than the windows hold.  512^3: 6.8 / 7.9 /
// 8.2 ms for stages 1 / 2 / 3 (3.3 to 4.4 TB/s where a copy does 4.8) against 11.4 / 12.8 / 11.4 ms
// of the fill-to-update chain of separate kernels; 256^3 0.91 / 1.04 / 1.06 ms against 1.6 / 1.8 / 1.7 ms.
//   A register spilled in the loop costs far more than its instructions: the reload waits for
// every DMA issued before it (stages 2 and 3 ran 13 ms at 512^3 with ten reloads per plane).
// Hence one-plane products instead of u, v, w windows, indices formed anew where they are used,
// and pin() and FENCE().  One wave per SIMD with 512 registers (32 x 8 tiles) ran
// 12.4 ms per stage at 512^3, opposite order of the z and the x, y parts in the two waves of a
// SIMD 7 % slower, LDS reads issued half a tap pair ahead no faster.
//   Wave priorities (phase 2) took 930 / 1040 / 1095 us for stages 1 / 2 / 3 at 256^3 where equal ones
// took 943 / 1051 / 1136; the younger wave first in phase 3 too, or always, was no faster.  LDS reads of the
// x taps issued a z tap ahead, lead() in phase 3, and the stage base loaded at the start of phase 3 were not
// faster either.  With the full chip running on a real flow the clock is at 2.05 GHz (2.35 on constant data).
//   Every value is computed by the reference's expression (-ffp-contract=off), so results are
// bit-identical to the reference cpu/ path.
#include <algorithm>
#include <type_traits>

#include "cns_fill.h"
#include "cns_runs.h"
#include "cns_stage_tile.h"

namespace cns {

namespace {

// where the arrays lie in LDS (the compiler's order, largest first)
constexpr int AT_DER = 0, AT_RAW = AT_DER + VNF * TILE * 8, AT_LEAD = AT_RAW + RNF * TILE * 8,
              AT_RING = AT_LEAD + LEAD * 8, AT_WZ = AT_RING + 8 * HALO * 8, AT_LV = AT_WZ + TILE * 8,
              AT_UX = AT_LV + LV * 8, AT_LU = AT_UX + LV * 8, AT_VY = AT_LU + LU * 8;

struct StageArgs {
    const double *base;  // U^n (stages 2 and 3)
    double *out;         // result (ghosted); must not alias cons
    double *q;           // primitives of the result (QOUT)
    double *d, *f;       // D and F (LAST)
    StepDt sd;           // the step's dt, made by stage 1 from the Courant maximum
    // WRAP, the box is its own periodic neighbour: stages 2 and 3 read cons at wrapped rows and planes,
    // of which stages 1 and 2 store the x ghosts with the result.  Stage 3 then also fills the
    // ghosts of cons and q: workgroups nt and above.
    int nt;
    Shell shell;
    double *fill_u;
};

// Stage 3 stores past the caches: its fifteen streams would push out the planes that the
// neighbours read again, and nothing reads them before the next step (8.37 -> 8.22 ms at 512^3, 1.08
// -> 1.06 at 256^3, 32.4 -> 31.8 us at 64^3).  What stages 1 and 2 store is read by the next one:
// stored so it made stage 2 2 to 4 % slower.
template <bool NT_>
__device__ __forceinline__ void put(double *p, unsigned off, double v)
{
    if (NT_)
        __builtin_nontemporal_store(v, &at(p, off));
    else
        at(p, off) = v;
}

template <bool STAGE1, bool LAST, bool QOUT, bool WRAP>
__global__ void __launch_bounds__(NT, 2)
stage_kernel(Geom g, const double *__restrict__ cons, StageArgs a, double dxi0, double dxi1, double dxi2,
             double eta, double alam, int kz, int ntx, int nty, BoxSet bs, int nbpb)
{
    __shared__ __align__(16) double raw[RNF * TILE];   // centre plane, raw
    // leading plane, raw: own cells; y halo's rho, my, mz (at LHY); x halo's rho, mx, mz (at LHX)
    __shared__ __align__(16) double s_lead[LEAD];
    __shared__ double der[VNF * TILE];                 // centre plane, derived
    __shared__ double s_lu[LU];                        // leading u: own rows, column c (0..39)
    __shared__ double s_lv[LV];                        // leading v: row r (0..R-1), column 4+c
    __shared__ double s_ux[LV];                        // row r (0..R-1), column 4+c
    __shared__ double s_vy[LU];                        // own rows, column c (0..39)
    __shared__ double s_wz[TILE];
    __shared__ double s_ring[8 * HALO];                // w of plane p on the halo columns, slot p % 8

    if (LAST && WRAP && (int)blockIdx.x >= a.nt) {
        const unsigned stride = (gridDim.x - a.nt) * NT;
        for (unsigned e = (blockIdx.x - a.nt) * NT + threadIdx.x; e < a.shell.total; e += stride)
            fill_cell<true>(g, a.shell, bs, 1, 1, 1, e, 0, a.fill_u, a.q, false);
        return;
    }
    int t = xcd_tile(blockIdx.x, a.nt);
    const int box = t / nbpb;
    t -= box * nbpb;
    cons += box * bs.su;
    const double *base = a.base + box * bs.su;
    double *out = a.out + box * bs.su;
    double *q = a.q + box * bs.sq, *dif = a.d + box * bs.sc, *flux = a.f + box * bs.sc;
    const int bx = t % ntx, by = (t / ntx) % nty, bz = t / (ntx * nty);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int gi0 = bx * TX, gj0 = by * BY;  // ghosted coordinates of tile cell (0, 0)
    const int kbeg = bz * kz, kend = min(kbeg + kz, g.n2);
    const int64_t cg = g.cg, pg = g.pg;
    // Stage 1 forms dt from the maximum (every workgroup for itself, the first one also for the
    // later stages and the host); stage 2 clears the maximum for the next step.
    double dt;
    if (STAGE1) {
        double courno;
        dt = courno_dt(a.sd.acc, a.sd.cfl, courno);
        if (blockIdx.x == 0 && threadIdx.x == 0) step_dt_store(a.sd, dt, courno);
    } else {
        dt = a.sd.dt[0];
        if (!LAST && blockIdx.x == 0 && threadIdx.x == 0) a.sd.acc[0] = 0ull;
    }
    const double ra = STAGE1 ? 0.0E0 : (LAST ? OneThird : ThreeQuarters);
    const double rb = STAGE1 ? 1.0E0 : (LAST ? TwoThirds : OneQuarter);
    const double dxi0s = dxi0 * dxi0, dxi1s = dxi1 * dxi1, dxi2s = dxi2 * dxi2;
    const unsigned xg = (unsigned)g.xg;

    // Shares of the halo cells, in units of one cell per lane: leading y halo, its ring and
    // wz on waves 0..3; leading x halo, its ring and wz on waves 4, 5; centre y halo and its
    // ux on waves 4..7; centre x halo on waves 0, 1; corners on wave 2; vy's x halo on 6, 7.
    // (The wave index is hidden at each use: the conditions, held across the loop, would be more
    // scalar registers than there are.)
    auto wv = [&]() {
        int w = wave;
        asm volatile("" : "+s"(w));
        return w;
    };

    // In-plane byte offset of tile cell (r, c)'s 16-byte pair, clamped into the array: cells
    // past the box feed discarded outputs only.
    // Row r of the tile in the array: clamped, and of a box that wraps the periodic image (a few
    // instructions that only the tiles at the box's y ends take; the conditions are formed where
    // they are used, like the wave's).
    auto row_of = [&](int r) {
        int j = min(gj0 + r, g.g1 - 1);
        if (WRAP && !STAGE1) {
            int j0 = gj0;
            asm volatile("" : "+s"(j0));
            if (j0 == 0 || j0 + R > g.g1 - NG) {
                j += j < NG ? g.n1 : 0;
                j -= j >= g.g1 - NG ? g.n1 : 0;
            }
        }
        return j;
    };
    auto plane_of = [&](int k) {  // ghosted plane index
        if (WRAP && !STAGE1) {
            k += k < NG ? g.n2 : 0;
            k -= k >= g.n2 + NG ? g.n2 : 0;
        }
        return (int64_t)k * pg;
    };
    auto pair_off = [&](int r, int c) {
        return (mul24(row_of(r), xg) + (unsigned)min(gi0 + c, g.xg - 2)) * 8u;
    };
    // the lane's cell in ghosted coordinates, whether it lies in the box, and its byte offset
    // within a ghosted plane
    struct Cell {
        int i, j;
        bool active;
        unsigned own8;
    };
    auto cell = [&]() {
        const unsigned tid = opaque_tid();
        Cell c;
        c.i = gi0 + (tid & (TX - 1)) + 4;
        c.j = gj0 + tid / TX + 4;
        c.active = c.i < g.n0 + NG && c.j < g.n1 + NG;
        c.own8 = (mul24(c.j, xg) + (unsigned)c.i) * 8u;
        return c;
    };
    auto issue_raw = [&](int k) {  // centre plane k: block `wave` of every field
        const double *p = cons + (int64_t)(k + NG) * pg;  // an interior plane
        const int w = wv();
        const unsigned lane = opaque_tid() & 63, e = 128 * w + 2 * lane;
        const unsigned off = pair_off(e / PX, e % PX);
        if (e < TILE) {
#pragma unroll
            for (int f = 0; f < RNF; f++) dma16(p + f * cg, off, (lds_double *)raw + f * TILE + 128 * w);
        }
    };
    // leading plane of centre plane k: own block wave % 4 of fields 0..2 (waves 0..3) or 3, 4;
    // the y halo's two blocks and the x halo's one on waves 4, 5, 6
    auto issue_lead = [&](int k) {
        const double *p = cons + plane_of(k + 2 * NG);
        const int w = wv();
        const unsigned lane = opaque_tid() & 63, ob = w & (OB - 1);
        const unsigned ooff = pair_off(4 + 4 * ob + (lane >> 4), 4 + 2 * (lane & 15));
        lds_double *l = (lds_double *)s_lead + 128 * ob;
        if (w < OB) {
            dma16(p, ooff, l);
            dma16(p + cg, ooff, l + NT);
            dma16(p + 2 * cg, ooff, l + 2 * NT);
        } else {
            dma16(p + 3 * cg, ooff, l + 3 * NT);
            dma16(p + 4 * cg, ooff, l + 4 * NT);
            if (w < 6) {  // rows 0..3 or BY+4..BY+7
                const unsigned hoff = pair_off((w == 4 ? 0 : BY + 4) + (lane >> 4), 4 + 2 * (lane & 15));
                lds_double *h = (lds_double *)s_lead + LHY + 128 * (w - 4);
                dma16(p, hoff, h);
                dma16(p + IMY * cg, hoff, h + YH);
                dma16(p + IMZ * cg, hoff, h + 2 * YH);
            } else if (w == 6) {  // columns 0..3 and TX+4..TX+7 of the own rows
                const int pr = lane & 3;
                const unsigned hoff = pair_off(4 + (lane >> 2), pr < 2 ? 2 * pr : 2 * pr + TX);
                lds_double *h = (lds_double *)s_lead + LHX;
                dma16(p, hoff, h);
                dma16(p + IMX * cg, hoff, h + XH);
                dma16(p + IMZ * cg, hoff, h + 2 * XH);
            }
        }
    };

    // Windows: plane k+m of the own column at [4+m].  wri is 1/rho, from which u, v, w of a
    // window plane are one product (ctoprim's own).
    double wmx[9], wmy[9], wmz[9], wE[9], wri[9], wp[9], wT[9], wux[9], wvy[9];

    // primitives of the leading plane: own cell into the windows' entry 8, u and v with their
    // halos into the lead tiles, w of the halo columns
    auto lead = [&]() {
        const double *area = s_lead;
        const unsigned tid = opaque_tid(), col = tid & (TX - 1), row = tid / TX;
        const double lr = area[tid];
        wmx[8] = area[RMX * NT + tid];
        wmy[8] = area[RMY * NT + tid];
        wmz[8] = area[RMZ * NT + tid];
        wE[8] = area[RE * NT + tid];
        double u_, v_, w_, eint;
        ctoprim_cell(lr, wmx[8], wmy[8], wmz[8], wE[8], u_, v_, w_, eint, wp[8]);
        wri[8] = 1.0E0 / lr;
        wT[8] = eint / CV;
        pin(wri[8], wp[8], wT[8]);
        s_lu[mul24(row, PX) + col + 4] = u_;
        s_lv[(row + 4) * TX + col] = v_;
        const int w = wv();
        if (w < 4) {
            const unsigned yr = row < 4 ? row : row + BY;  // waves 0..3: rows 0..7
            const double hinv = 1.0E0 / area[LHY + tid];
            s_lv[yr * TX + col] = area[LHY + YH + tid] * hinv;
            s_wz[mul24(yr, PX) + col + 4] = area[LHY + 2 * YH + tid] * hinv;
        }
        if (w == 4 || w == 5) {
            const unsigned xid = tid & 127, c8 = xid & 7;
            const double hinv = 1.0E0 / area[LHX + xid];
            const unsigned l = mul24(xid >> 3, PX) + (c8 < 4 ? c8 : c8 + TX);
            s_lu[l] = area[LHX + XH + xid] * hinv;
            s_wz[l + 4 * PX] = area[LHX + 2 * XH + xid] * hinv;
        }
    };
    auto shift = [&]() {
#pragma unroll
        for (int m = 0; m < 8; m++) {
            wmx[m] = wmx[m + 1]; wmy[m] = wmy[m + 1]; wmz[m] = wmz[m + 1]; wE[m] = wE[m + 1];
            wri[m] = wri[m + 1]; wp[m] = wp[m + 1]; wT[m] = wT[m + 1];
            wux[m] = wux[m + 1]; wvy[m] = wvy[m + 1];
        }
    };

    // ux, vy of the leading plane into the windows; w of the halo columns: planes k .. k+7 are
    // in the ring, k+8 where lead() left it, which gives wz there and then takes the place of plane k
    auto lead_grads = [&](int k) {
        const unsigned tid = opaque_tid(), col = tid & (TX - 1), row = tid / TX;
        double a[9], b[9];
        {
            const Taps<AT_LU> p_lu(s_lu, mul24(row, PX) + col);
            const Taps<AT_LV> p_lv(s_lv, tid);
#pragma unroll
            for (int m = 0; m < 9; m++)
                if (m != 4) {
                    a[m] = p_lu[m];
                    b[m] = p_lv[m * TX];
                }
            FENCE();
        }
#define LUX(mm) a[4 + (mm)]
#define LVY(mm) b[4 + (mm)]
        wux[8] = D1(LUX) * dxi0;
        wvy[8] = D1(LVY) * dxi1;
#undef LUX
#undef LVY
        pin(wux[8], wvy[8]);
        FENCE();
        const int w = wv();
        if (w < 6) {
            const unsigned xid = tid & 127, c8 = xid & 7;
            const unsigned rc = w < 4 ? tid : YH + xid;
            const unsigned l = w < 4 ? mul24(row < 4 ? row : row + BY, PX) + col + 4
                               : mul24((xid >> 3) + 4, PX) + (c8 < 4 ? c8 : c8 + TX);
            const Taps<0> p_r(s_ring, rc);  // (slots are scalars: the place goes with them)
            a[8] = s_wz[l];  // w of plane k+8, left here by lead()
#pragma unroll
            for (int m = 0; m < 8; m++)
                if (m != 4) a[m] = p_r[((k + m) & 7) * HALO];
            FENCE();
#define RW(mm) a[4 + (mm)]
            s_wz[l] = D1(RW) * dxi2;
#undef RW
            s_ring[(k & 7) * HALO + rc] = a[8];
        }
    };

    // Fill the windows and the ring with planes kbeg .. kbeg+7: all their loads at once, into
    // the windows' own registers, then the primitives of all eight planes with their u and v
    // rows and columns in LDS (the centre plane's DMA meanwhile has the raw tile), then ux and vy.
    // Its time is the loads' latency and the arithmetic of eight planes of primitives, about 9 us;
    // plane by plane through the staged tile, with sixteen barriers, it took 15 (a stage of 16^3
    // 23 -> 18 us, of 64^3 42 -> 32 us, of 130 x 97 x 61 95 -> 85 us).
    {
        // where plane kbeg+m's u rows and v columns are until ux and vy are formed
        double *const lu[8] = {s_lead, s_lead + LU, s_lead + 2 * LU, s_lead + 3 * LU, s_lu, s_ux, s_vy, s_wz};
        double *const lv[8] = {s_lead + 4 * LU, s_lv, der, der + LV, der + 2 * LV, der + 3 * LV, der + 4 * LV,
                               der + 5 * LV};
        const unsigned tid = opaque_tid(), col = tid & (TX - 1), row = tid / TX;
        const unsigned xid = tid & 127, c8 = xid & 7, xcol = c8 < 4 ? c8 : c8 + TX, yrow = row < 4 ? row : row + BY;
        const bool yl = wave < 4, halo = wave < 6;
        double hr[8], hm[8], hz[8];
        {
            auto off8 = [&](unsigned r, unsigned c) {
                return (mul24(row_of((int)r), xg) + (unsigned)min(gi0 + (int)c, g.xg - 1)) * 8u;
            };
            const unsigned own8 = off8(row + 4, col + 4), h8 = yl ? off8(yrow, col + 4) : off8((xid >> 3) + 4, xcol);
#pragma unroll
            for (int m = 0; m < 8; m++) {
                const double *p = cons + plane_of(kbeg + m);
                wri[m] = at(p, own8);
                wmx[m] = at(p + IMX * cg, own8);
                wmy[m] = at(p + IMY * cg, own8);
                wmz[m] = at(p + IMZ * cg, own8);
                wE[m] = at(p + IENE * cg, own8);
                hr[m] = hm[m] = hz[m] = 1.0;
                if (halo) {
                    hr[m] = at(p, h8);
                    hm[m] = at(p + (yl ? IMY : IMX) * cg, h8);
                    hz[m] = at(p + IMZ * cg, h8);
                }
            }
        }
        issue_raw(kbeg);
        FENCE();
#pragma unroll
        for (int m = 0; m < 8; m++) {
            double u_, v_, w_, eint;
            const double rho = wri[m];
            ctoprim_cell(rho, wmx[m], wmy[m], wmz[m], wE[m], u_, v_, w_, eint, wp[m]);
            wri[m] = 1.0E0 / rho;
            wT[m] = eint / CV;
            pin(wri[m], wp[m], wT[m]);
            lu[m][mul24(row, PX) + col + 4] = u_;
            lv[m][(row + 4) * TX + col] = v_;
            if (halo) {
                const double hinv = 1.0E0 / hr[m];
                if (yl)
                    lv[m][yrow * TX + col] = hm[m] * hinv;
                else
                    lu[m][mul24(xid >> 3, PX) + xcol] = hm[m] * hinv;
                s_ring[((kbeg + m) & 7) * HALO + (yl ? tid : YH + xid)] = hz[m] * hinv;
            }
            FENCE();
        }
        __syncthreads();
        auto grads = [&](int m) {
            lds_tap<double> *p_lu = (lds_tap<double> *)lu[m] + mul24(row, PX) + col + 4, *p_lv = (lds_tap<double> *)lv[m] + (row + 4) * TX + col;
#define LUX(mm) p_lu[mm]
#define LVY(mm) p_lv[(mm) * TX]
            wux[m] = D1(LUX) * dxi0;
            wvy[m] = D1(LVY) * dxi1;
#undef LUX
#undef LVY
            pin(wux[m], wvy[m]);
            FENCE();
        };
#pragma unroll
        for (int m = 0; m < 4; m++) grads(m);
        __syncthreads();  // the planes in s_lead are used
        issue_lead(kbeg);
#pragma unroll
        for (int m = 4; m < 8; m++) grads(m);
        __builtin_amdgcn_s_waitcnt(0xF70);
        __syncthreads();
    }

#pragma unroll 1
    for (int k = kbeg; k < kend; k++) {
        const double *d_u = der + VU * TILE, *d_v = der + VV * TILE, *d_w = der + VW * TILE, *d_t = der + VT * TILE,
                     *d_p = der + VP * TILE;
        // ---------------- phase 1: primitives of the leading plane, derived tiles of the centre plane
        lead();
        {
            const unsigned tid = opaque_tid(), col = tid & (TX - 1), row = tid / TX, lane = tid & 63;
            const unsigned me = mul24(row + 4, PX) + col + 4;
            der[VU * TILE + me] = wmx[4] * wri[4];
            der[VV * TILE + me] = wmy[4] * wri[4];
            der[VW * TILE + me] = wmz[4] * wri[4];
            der[VT * TILE + me] = wT[4];
            der[VP * TILE + me] = wp[4];
            auto halo_prim = [&](unsigned l) {
                double u_, v_, w_, eint, p_;
                ctoprim_cell(raw[RRHO * TILE + l], raw[RMX * TILE + l], raw[RMY * TILE + l], raw[RMZ * TILE + l],
                             raw[RE * TILE + l], u_, v_, w_, eint, p_);
                der[VU * TILE + l] = u_;
                der[VV * TILE + l] = v_;
                der[VW * TILE + l] = w_;
                der[VT * TILE + l] = eint / CV;
                der[VP * TILE + l] = p_;
            };
            const int w = wv();
            if (w >= 4) {
                const unsigned yrow = row - 8;
                halo_prim(mul24(yrow < 4 ? yrow : yrow + BY, PX) + col + 4);
            }
            if (w < 2) {
                const unsigned c8 = tid & 7;
                halo_prim(mul24((tid >> 3) + 4, PX) + (c8 < 4 ? c8 : c8 + TX));
            }
            if (w == 2) {  // u and v only
                const unsigned r8 = lane >> 3, c8 = lane & 7;
                const unsigned l = mul24(r8 < 4 ? r8 : r8 + BY, PX) + (c8 < 4 ? c8 : c8 + TX);
                const double cinv = 1.0E0 / raw[RRHO * TILE + l];
                der[VU * TILE + l] = raw[RMX * TILE + l] * cinv;
                der[VV * TILE + l] = raw[RMY * TILE + l] * cinv;
            }
        }
        __syncthreads();  // B

        // ---------------- phase 2
        // Of the two waves of a SIMD the older wins every choice, and would wait at C while the
        // younger (4..7) runs alone: the younger goes first up to the end of the z terms.
        if (wave >= 4) __builtin_amdgcn_s_setprio(1);
        if (k + 1 < kend) issue_lead(k + 1);
        double F[5], zf[5], rho_c;
        lead_grads(k);
        {
            const unsigned tid = opaque_tid(), col = tid & (TX - 1), row = tid / TX;
            const unsigned me = mul24(row + 4, PX) + col + 4;
            {
                // ux, vy, wz of the centre plane: own cells from the windows, the halos the mixed
                // derivatives read from the derived tiles (cpu/diffterm.cpp:77-151)
                s_ux[(row + 4) * TX + col] = wux[4];
                const int w = wv();
                if (w >= 4) {
                    const unsigned yrow = row - 8, yr = yrow < 4 ? yrow : yrow + BY;
                    const Taps<AT_DER> p_u(d_u, mul24(yr, PX) + col);
                    double a[9];
#pragma unroll
                    for (int m = 0; m < 9; m++)
                        if (m != 4) a[m] = p_u[m];
                    FENCE();
#define CUX(mm) a[4 + (mm)]
                    s_ux[yr * TX + col] = D1(CUX) * dxi0;
#undef CUX
                }
                s_vy[mul24(row, PX) + col + 4] = wvy[4];
                if (w >= 6) {
                    const unsigned xid = tid & 127, c8 = xid & 7, l = mul24(xid >> 3, PX) + (c8 < 4 ? c8 : c8 + TX);
                    const Taps<AT_DER> p_v(d_v, l);
                    double a[9];
#pragma unroll
                    for (int m = 0; m < 9; m++)
                        if (m != 4) a[m] = p_v[m * PX];
                    FENCE();
#define CVY(mm) a[4 + (mm)]
                    s_vy[l] = D1(CVY) * dxi1;
#undef CVY
                }
                rho_c = raw[RRHO * TILE + me];
            }
            FENCE();
        }
        double zx = 0.0, zy = 0.0, zz = 0.0, zt = 0.0, uz = 0.0, vz = 0.0, mz = 0.0;
        {
            // every z term of the cell, from the windows
            double hs[5], uxz, vyz, wzc;
            zx = CENTER * (wmx[4] * wri[4]);
            zy = CENTER * (wmy[4] * wri[4]);
            zz = CENTER * (wmz[4] * wri[4]);
            zt = CENTER * wT[4];
#define ZTAP(m, C1, C2, FIRST)                                                                                   \
    {                                                                                                            \
        const double w1 = wmz[4 + m] * wri[4 + m], w0 = wmz[4 - m] * wri[4 - m];                                 \
        hyp_tap<FIRST>(C1, wmz[4 + m], wmz[4 - m], wmx[4 + m], wmx[4 - m], wmy[4 + m], wmy[4 - m], wE[4 + m],     \
                       wE[4 - m], wp[4 + m], wp[4 - m], wp[4 + m], wp[4 - m], w1, w0, hs);                                             \
        tap<FIRST>(wzc, C1 * (w1 - w0));                                                                         \
        tap<false>(zz, C2 * (w1 + w0));                                                                          \
        const double u1 = wmx[4 + m] * wri[4 + m], u0 = wmx[4 - m] * wri[4 - m];                                 \
        tap<FIRST>(uz, C1 * (u1 - u0));                                                                          \
        tap<false>(zx, C2 * (u1 + u0));                                                                          \
        const double v1 = wmy[4 + m] * wri[4 + m], v0 = wmy[4 - m] * wri[4 - m];                                 \
        tap<FIRST>(vz, C1 * (v1 - v0));                                                                          \
        tap<false>(zy, C2 * (v1 + v0));                                                                          \
        tap<false>(zt, C2 * (wT[4 + m] + wT[4 - m]));                                                            \
        tap<FIRST>(uxz, C1 * (wux[4 + m] - wux[4 - m]));                                                         \
        tap<FIRST>(vyz, C1 * (wvy[4 + m] - wvy[4 - m]));                                                         \
        pin(hs[0], hs[1], hs[2], hs[3], hs[4], wzc, zz, uz, zx, vz, zy, zt, uxz, vyz);                            \
        FENCE();                                                                                                 \
    }
            ZTAP(1, ALP, OFF1, true)
            ZTAP(2, BET, OFF2, false)
            ZTAP(3, GAM, OFF3, false)
            ZTAP(4, DEL, OFF4, false)
#undef ZTAP
            zf[IRHO] = hs[0] * dxi2;
            zf[IMZ] = hs[1] * dxi2;
            zf[IMX] = hs[2] * dxi2;
            zf[IMY] = hs[3] * dxi2;
            zf[IENE] = hs[4] * dxi2;
            wzc = wzc * dxi2;
            uz = uz * dxi2;
            vz = vz * dxi2;
            zx = zx * dxi2s;
            zy = zy * dxi2s;
            zz = zz * dxi2s;
            zt = zt * dxi2s;
            mz = uxz * dxi2 + vyz * dxi2;
            pin(zf[0], zf[1], zf[2], zf[3], zf[4], uz, vz, zx, zy, zz, zt, mz);
            FENCE();
            const unsigned tid = opaque_tid();
            s_wz[mul24(tid / TX + 4, PX) + (tid & (TX - 1)) + 4] = wzc;
        }
        __builtin_amdgcn_s_setprio(0);
        shift();  // the centre plane is window entry 3 from here
        {
            // from four rows above the own cell: every tap is a non-negative constant away
            const unsigned tid = opaque_tid(), me4 = mul24(tid / TX, PX) + (tid & (TX - 1)) + 4;
            const Taps<AT_RAW> s_c(raw, me4);
            const Taps<AT_DER> s_d(der, me4);
            double hs[5], A[12];
            // fields n, a, b, E of the raw tile, p and v of the derived one at taps +o and -o
            constexpr int Z = 4 * PX;
            auto load = [&](double (&T)[12], int n, int a_, int b_, int v, int o) {
                T[0] = s_c[n * TILE + Z + o]; T[1] = s_c[n * TILE + Z - o];
                T[2] = s_c[a_ * TILE + Z + o]; T[3] = s_c[a_ * TILE + Z - o];
                T[4] = s_c[b_ * TILE + Z + o]; T[5] = s_c[b_ * TILE + Z - o];
                T[6] = s_c[RE * TILE + Z + o]; T[7] = s_c[RE * TILE + Z - o];
                T[8] = s_d[VP * TILE + Z + o]; T[9] = s_d[VP * TILE + Z - o];
                T[10] = s_d[v * TILE + Z + o]; T[11] = s_d[v * TILE + Z - o];
            };
#define HT(FIRST, C, T) \
    hyp_tap<FIRST>(C, T[0], T[1], T[2], T[3], T[4], T[5], T[6], T[7], T[8], T[9], T[8], T[9], T[10], T[11], hs); \
    pin(hs[0], hs[1], hs[2], hs[3], hs[4]); FENCE()
            load(A, RMX, RMY, RMZ, VU, 1); FENCE();
            HT(true, ALP, A);
            load(A, RMX, RMY, RMZ, VU, 2); FENCE();
            HT(false, BET, A);
            load(A, RMX, RMY, RMZ, VU, 3); FENCE();
            HT(false, GAM, A);
            load(A, RMX, RMY, RMZ, VU, 4); FENCE();
            HT(false, DEL, A);
            F[IRHO] = -(hs[0]) * dxi0;
            F[IMX] = -(hs[1]) * dxi0;
            F[IMY] = -(hs[2]) * dxi0;
            F[IMZ] = -(hs[3]) * dxi0;
            F[IENE] = -(hs[4]) * dxi0;
            load(A, RMY, RMX, RMZ, VV, PX); FENCE();
            HT(true, ALP, A);
            load(A, RMY, RMX, RMZ, VV, 2 * PX); FENCE();
            HT(false, BET, A);
            load(A, RMY, RMX, RMZ, VV, 3 * PX); FENCE();
            HT(false, GAM, A);
            load(A, RMY, RMX, RMZ, VV, 4 * PX); FENCE();
            HT(false, DEL, A);
#undef HT
            F[IRHO] = F[IRHO] - hs[0] * dxi1;
            F[IMY] = F[IMY] - hs[1] * dxi1;
            F[IMX] = F[IMX] - hs[2] * dxi1;
            F[IMZ] = F[IMZ] - hs[3] * dxi1;
            F[IENE] = F[IENE] - hs[4] * dxi1;
#pragma unroll
            for (int l = 0; l < NC; l++) F[l] = F[l] - zf[l];
            pin(F[0], F[1], F[2], F[3], F[4], rho_c);
        }
        __syncthreads();  // C

        // ---------------- phase 3
        const int64_t zk = (int64_t)(k + NG) * pg;
        if (k + 1 < kend) issue_raw(k + 1);
        {   // held in the lead tiles' own cells (read by the neighbours before C) until the update
            const unsigned tid = opaque_tid(), col = tid & (TX - 1), row = tid / TX;
            s_lu[mul24(row, PX) + col + 4] = rho_c;
            s_lv[(row + 4) * TX + col] = F[IENE];
        }
        {
            // diffterm's x and y terms, from the tiles, then its sums as the reference forms them
            // (cpu/diffterm.cpp:159-311)
            const unsigned tid = opaque_tid(), col = tid & (TX - 1), row = tid / TX;
            const unsigned me4 = mul24(row, PX) + col + 4;  // as above
            const Taps<AT_DER> s_d(der, me4);
            const Taps<AT_WZ> s_z(s_wz, me4);
            constexpr int Z = 4 * PX;
            double A[12], xu, xv, xw, xt, d2v, d2w, m1, m2;
            // u, v, w, T of the derived tile, wz and vy at taps +o and -o in x
            const Taps<AT_VY> s_m4(s_vy, me4 - 4);
            auto load = [&](double (&T)[12], int o) {
                T[0] = s_d[VU * TILE + Z + o]; T[1] = s_d[VU * TILE + Z - o];
                T[2] = s_d[VV * TILE + Z + o]; T[3] = s_d[VV * TILE + Z - o];
                T[4] = s_d[VW * TILE + Z + o]; T[5] = s_d[VW * TILE + Z - o];
                T[6] = s_d[VT * TILE + Z + o]; T[7] = s_d[VT * TILE + Z - o];
                T[8] = s_z[Z + o]; T[9] = s_z[Z - o];
                T[10] = s_m4[4 + o]; T[11] = s_m4[4 - o];
            };
            // second differences of u, v, w, T; first of T[2 * f] (d2v), w (d2w), and of the two mixed terms
#define DT(FIRST, C1, C2, T, f)                  \
    tap<false>(xu, C2 * (T[0] + T[1]));          \
    tap<false>(xv, C2 * (T[2] + T[3]));          \
    tap<false>(xw, C2 * (T[4] + T[5]));          \
    tap<false>(xt, C2 * (T[6] + T[7]));          \
    tap<FIRST>(d2v, C1 * (T[2 * f] - T[2 * f + 1])); \
    tap<FIRST>(d2w, C1 * (T[4] - T[5]));         \
    tap<FIRST>(m1, C1 * (T[10] - T[11]));        \
    tap<FIRST>(m2, C1 * (T[8] - T[9]));          \
    pin(xu, xv, xw, xt, d2v, d2w, m1, m2);       \
    FENCE()
            xu = CENTER * (wmx[3] * wri[3]); xv = CENTER * (wmy[3] * wri[3]);
            xw = CENTER * (wmz[3] * wri[3]); xt = CENTER * wT[3];
            load(A, 1); FENCE();
            DT(true, ALP, OFF1, A, 1);
            load(A, 2); FENCE();
            DT(false, BET, OFF2, A, 1);
            load(A, 3); FENCE();
            DT(false, GAM, OFF3, A, 1);
            load(A, 4); FENCE();
            DT(false, DEL, OFF4, A, 1);
            double sx = FourThirds * (xu * dxi0s), sy = xv * dxi0s, sz = xw * dxi0s, st = xt * dxi0s;
            const double vx = d2v * dxi0, wx = d2w * dxi0, mx = m1 * dxi0 + m2 * dxi0;
            pin(sx, sy, sz, st);
            double rkb[5];
            if (!STAGE1) {  // (cells past the box read clamped, for nothing: no divergent branch here)
                const unsigned t3 = opaque_tid();
                const unsigned off = (mul24(min(gj0 + (int)(t3 / TX) + 4, g.g1 - 1), xg)
                                      + (unsigned)min(gi0 + (int)(t3 & (TX - 1)) + 4, g.g0 - 1)) * 8u;
#pragma unroll
                for (int l = 0; l < NC; l++) rkb[l] = at(base + l * cg + zk, off);
            }
            xu = CENTER * (wmx[3] * wri[3]); xv = CENTER * (wmy[3] * wri[3]);
            xw = CENTER * (wmz[3] * wri[3]); xt = CENTER * wT[3];
            const Taps<AT_UX> s_n(s_ux, tid);
            auto ytap = [&](auto first, double c1, double c2, int o, int on) {
                constexpr bool FI = decltype(first)::value;
                {
                    const double u1 = s_d[VU * TILE + Z + o], u0 = s_d[VU * TILE + Z - o], v1 = s_d[VV * TILE + Z + o],
                                 v0 = s_d[VV * TILE + Z - o], w1 = s_d[VW * TILE + Z + o], w0 = s_d[VW * TILE + Z - o];
                    FENCE();
                    tap<false>(xu, c2 * (u1 + u0));
                    tap<false>(xv, c2 * (v1 + v0));
                    tap<false>(xw, c2 * (w1 + w0));
                    tap<FI>(d2v, c1 * (u1 - u0));
                    tap<FI>(d2w, c1 * (w1 - w0));
                    pin(xu, xv, xw, d2v, d2w);
                    FENCE();
                }
                {
                    const double t1 = s_d[VT * TILE + Z + o], t0 = s_d[VT * TILE + Z - o], z1 = s_z[Z + o], z0 = s_z[Z - o],
                                 n1 = s_n[4 * TX + on], n0 = s_n[4 * TX - on];
                    FENCE();
                    tap<false>(xt, c2 * (t1 + t0));
                    tap<FI>(m1, c1 * (n1 - n0));
                    tap<FI>(m2, c1 * (z1 - z0));
                    pin(xt, m1, m2);
                    FENCE();
                }
            };
            ytap(std::true_type(), ALP, OFF1, PX, TX);
            ytap(std::false_type(), BET, OFF2, 2 * PX, 2 * TX);
            ytap(std::false_type(), GAM, OFF3, 3 * PX, 3 * TX);
            ytap(std::false_type(), DEL, OFF4, 4 * PX, 4 * TX);
#undef DT
            sx = sx + xu * dxi1s;
            sy = sy + FourThirds * (xv * dxi1s);
            sz = sz + xw * dxi1s;
            st = st + xt * dxi1s;
            const double tauxy = d2v * dxi1 + vx, wy = d2w * dxi1, my = m1 * dxi1 + m2 * dxi1;
            const double uzz = zx, vzz = zy, wzz = zz, tzz = zt;
            double D[5];
            D[IRHO] = 0.0E0;
            D[IMX] = eta * (sx + uzz + OneThird * mx);
            D[IMY] = eta * (sy + vzz + OneThird * my);
            D[IMZ] = eta * (sz + FourThirds * wzz + OneThird * mz);
            {
                const double ux = wux[3], vy = wvy[3], wz = s_z[Z];
                const double divu = TwoThirds * (ux + vy + wz);
                const double tauxx = 2.E0 * ux - divu;
                const double tauyy = 2.E0 * vy - divu;
                const double tauzz = 2.E0 * wz - divu;
                const double tauxz = uz + wx;
                const double tauyz = vz + wy;
                double mechwork = tauxx * ux + tauyy * vy + tauzz * wz + (tauxy * tauxy) + (tauxz * tauxz)
                                  + (tauyz * tauyz);
                mechwork = eta * mechwork + D[IMX] * (wmx[3] * wri[3]) + D[IMY] * (wmy[3] * wri[3])
                           + D[IMZ] * (wmz[3] * wri[3]);
                D[IENE] = alam * (st + tzz) + mechwork;
            }
            rho_c = s_lu[mul24(row, PX) + col + 4];
            F[IENE] = s_lv[(row + 4) * TX + col];
            const double uc[5] = {rho_c, wmx[3], wmy[3], wmz[3], wE[3]};
            // the centre plane's DMA has landed before the stores join the queue, so the barrier
            // that ends the phase need not wait for them
            __builtin_amdgcn_s_waitcnt(0xF70);
            const Cell c = cell();
            if (c.active) {
                const unsigned own8 = c.own8,
                               int8 = (mul24(c.j - NG, g.x) + (unsigned)(c.i - NG)) * 8u;
                const int64_t fk = (int64_t)k * g.p;
                double o[5];
#pragma unroll
                for (int l = 0; l < NC; l++) {
                    if (LAST) {
                        put<true>(dif + l * g.c + fk, int8, D[l]);
                        put<true>(flux + l * g.c + fk, int8, F[l]);
                    }
                    // STAGE1: cons + dt(D+F) (cpu/advance.cpp:82); then ra*base + rb*(cons + dt(D+F))
                    // (:114-116, :148-150)
                    o[l] = STAGE1 ? uc[l] + dt * (D[l] + F[l]) : ra * rkb[l] + rb * (uc[l] + dt * (D[l] + F[l]));
                    put<LAST>(out + l * cg + zk, own8, o[l]);
                }
                // the x ghosts that are images of the cell
                int i0 = gi0;
                asm volatile("" : "+s"(i0));
                if (WRAP && !LAST && (i0 == 0 || i0 + TX + NG > g.n0)) {
                    const unsigned n8 = (unsigned)g.n0 * 8u;
                    if (c.i < 2 * NG) {
#pragma unroll
                        for (int l = 0; l < NC; l++) at(out + l * cg + zk, own8 + n8) = o[l];
                    }
                    if (c.i >= g.n0) {
#pragma unroll
                        for (int l = 0; l < NC; l++) at(out + l * cg + zk, own8 - n8) = o[l];
                    }
                }
                if (QOUT) {  // cpu/ctoprim.cpp:23-38
                    double u, v, w, eint, p;
                    ctoprim_cell(o[IRHO], o[IMX], o[IMY], o[IMZ], o[IENE], u, v, w, eint, p);
                    double *qk = q + zk;
                    at(qk, own8) = o[IRHO];
                    at(qk + QU * cg, own8) = u;
                    at(qk + QV * cg, own8) = v;
                    at(qk + QW * cg, own8) = w;
                    at(qk + QPRES * cg, own8) = p;
                    at(qk + QTEMP * cg, own8) = eint / CV;
                }
            }
        }
        __syncthreads();  // A
    }
}

// z runs.  A CU holds one workgroup, so a launch takes ceil(workgroups / 256) rounds of
// (planes + the window fill and launch, which cost about kFill planes: 11 us of 6.7 us a plane); the run
// length that makes this smallest is taken.
constexpr int kCUs = 256;
constexpr double kFill = 1.6;

int stage_kz(const Geom &g, int64_t tiles) { return stage_run(g.n2, tiles, kCUs, kFill); }

}  // namespace

bool stage_fits(const Geom &g)
{
    return g.pg < (1 << 29) && g.xg < (1 << 24) && g.g1 < (1 << 24);
}

// A tile of 32 x 16 cells costs its time however few of them the box has, so a tall column of a few
// cells is stepped faster by the separate kernels, whose tiles are half as high: us a step with one
// kernel a stage / separate kernels, 4 x 4 x 512 112 / 168, x 4096 395 / 337, x 20000 1689 / 1360;
// 8 x 8 x 512 109 / 175, x 4096 401 / 393, x 20000 1747 / 1647; 16 x 8 x 20000 2053 / 2650, 12 x 12 x 20000
// 2255 / 3806.
bool stage_pays(const Geom &g) { return g.n0 > 8 || g.n1 > 8 || g.n2 < 16 * kCUs; }

// Reading at wrapped addresses and storing the x ghosts beside the result costs a plane about
// 1.5 % (scalar registers that no longer fit), two fill launches their time and two gaps: a step
// with / without them takes 73 / 80 us at 16^3, 113 / 120 at 64^3, 466 / 480 at 128^3, 3.24 / 3.26
// ms at 256^3 (128 planes a CU), 6.53 / 6.58 at 320^3 (250), 25.9 / 25.6 at 512^3 (1024).
bool stage_wraps(const Geom &g)
{
    return (int64_t)((g.n0 + TX - 1) / TX) * ((g.n1 + BY - 1) / BY) * g.n2 <= 512 * kCUs;
}

hipError_t launch_stage(const Geom &g, const double *cons, const double *base, double *out, double *q, double *d,
                        double *f, const StepDt &sd, const double dxi[3], double eta, double alam, int phase,
                        hipStream_t s, const BoxSet &bs, double *wrapped)
{
    if (bs.n < 1 || !stage_fits(g) || (wrapped && bs.n != 1)) return hipErrorInvalidValue;
    const int ntx = (g.n0 + TX - 1) / TX, nty = (g.n1 + BY - 1) / BY;
    const int kz = stage_kz(g, (int64_t)ntx * nty * bs.n);
    const int64_t nbpb = (int64_t)ntx * nty * ((g.n2 + kz - 1) / kz);
    if (nbpb * bs.n > 0x7fffffff) return hipErrorInvalidValue;
    const int nt = (int)(nbpb * bs.n);
    const StageArgs a{base, out, q, d, f, sd, nt, make_shell(g, kOneBox), wrapped};
    // Ghost cells of stage 3, about one a thread in a small box, whose fill workgroups take the
    // CUs that the stage leaves idle; at most one workgroup a CU.
    int nb = nt;
    if (wrapped && phase == 3) {
        const int64_t total = shell_cells(g);
        if (total > 0xffffffffll - kCUs * NT) return hipErrorInvalidValue;
        nb += (int)std::min<int64_t>((total + NT - 1) / NT, kCUs);
    }
#define STAGE(S1, L, QO)                                                                                           \
    if (wrapped)                                                                                                   \
        stage_kernel<S1, L, QO, true><<<nb, NT, 0, s>>>(g, cons, a, dxi[0], dxi[1], dxi[2], eta, alam, kz, ntx, nty, \
                                                        bs, (int)nbpb);                                            \
    else                                                                                                           \
        stage_kernel<S1, L, QO, false><<<nb, NT, 0, s>>>(g, cons, a, dxi[0], dxi[1], dxi[2], eta, alam, kz, ntx,     \
                                                         nty, bs, (int)nbpb)
    switch (phase) {
    case 1: STAGE(true, false, false); break;
    case 2: STAGE(false, false, true); break;
    case 3: STAGE(false, true, false); break;
    default: return hipErrorInvalidValue;
    }
#undef STAGE
    return hipGetLastError();
}

}  // namespace cns
