// cns_batch_stage.hip -- one RK stage of the batched engine's 32-wide boxes in a single
// z-marching kernel (gfx950).
//
// The stage kernel of the plain step (cns_stage.hip: its windows, tiles, phases and LDS
// staging) for ghost-free boxes and both flux types: a workgroup takes a 32 x 16 column tile
// (FP32 flux: or 32 x 24) and a run of planes of one box and produces, from the five conserved fields alone, the
// result of the stage; in stage 3 also the Courant maximum of the result.  The separate
// kernels (cns_batch.hip) pass Q, wz and D through memory between a wz, a diffterm and a
// hypterm launch.
//
// What differs from cns_stage.hip.
//   Periodic rows.  Halos lie at wrapped addresses and rows of odd edges are 8-byte aligned,
// so planes are staged by direct-to-LDS loads of 4 bytes a lane: 32 cells of one row each, at
// a scalar row offset and one wrapped lane offset, and the x halos (four rows of eight cells)
// at a second one.
//   The centre plane's own cells come from the windows, so only its halo is loaded.
//   Flux type FT.  Primitives, the update and the Courant number are FP64 in both modes; with
// FT = float the windows and tiles hold the rounded values (u, v, w too, which FP64 recomputes
// as one product) and the pressure less the box's reference, as the separate kernels' fields.
//   FP32 flux: tall tiles.  A wave issues an instruction every four cycles at best and waits half
// its time, whatever the type, so a plane of FP32 took as long as one of FP64.  Its windows are
// half the size, though: 168 registers a lane and 143 KB of LDS hold three waves a SIMD, 32 x 24
// cells a plane at 1.35 times the time of 32 x 16 (G cell-steps/s, one height for all: edge 96 6.5
// -> 7.3, 48 5.1 -> 6.0, 24 3.7 -> 5.6).  A box's rows are covered by both heights (fused_list()),
// for which the kernel holds both bodies; waves 8..11 end at once in a short tile.  64 boxes x4
// 10.4 -> 9.35 ms, serving 40 boxes x8 40.1 -> 36.4 ms; 24 rows alone gave 9.7 and 37.7.
//   Every value is the separate kernels' expression: the same bits, and in FP64 the reference's.
#include "cns_batch_dev.h"
#include "cns_stage_tile.h"
#include "cns_stencil_ops.h"

namespace cns {

namespace {

constexpr int CORN = 64;  // corner cells of a tile

// A tile of BY rows: cns_stage_tile.h's sizes for them, and who does what.
template <typename FT, int BY_>
struct Rows {
    static constexpr bool F32 = sizeof(FT) == 4;
    static constexpr int BY = BY_, R = BY + 8, NT = TX * BY, NW = NT / 64;
    static constexpr int TILE = R * PX, XH = 8 * BY, HALO = YH + XH;
    static constexpr int LHY = 5 * NT, LHX = LHY + 3 * YH, LEAD = LHX + 3 * XH, LU = BY * PX, LV = R * TX;
    static_assert(LEAD * 8 >= (4 * LU + LV) * (int)sizeof(FT) && 5 * TILE >= 6 * LV && TILE >= LU && LV >= LU,
                  "places of the window fill");
    // Shares of the halo cells, one cell per lane, as first waves: leading y halo, its ring and wz
    // on waves 0..3; leading x halo, its ring and wz on XW waves from 4; centre y halo and its ux on
    // four from YC; centre x halo on XW from XC; corners on wave CC; vy's x halo on XW from VX.
    static constexpr int XW = XH / 64, YC = NW - 4, XC = BY == 16 ? 0 : 5, CC = BY == 16 ? 2 : 4, VX = BY == 16 ? 6 : 5;
    // staged x halo: XS waves of 32 cells, then two of corners
    static constexpr int XS = XH / 32;
    static_assert(XH % 64 == 0 && NW >= 8 && 4 + XW <= NW && XC + XW <= NW && VX + XW <= NW && XS + 2 <= NW, "wave shares");
    // staged FP64 halo of the centre plane: y halo (rho; FP32 flux: all five fields, which FP64
    // loads into the tile itself), x halo of five fields, corners of rho, mx, my
    static constexpr int HX = (F32 ? 5 : 1) * YH, HC = HX + 5 * XH, H = HC + 3 * CORN;
};
// The largest tile, whose arrays every tile uses, and where they lie in LDS (the compiler's order,
// largest first)
template <typename FT>
struct Lay : Rows<FT, sizeof(FT) == 4 ? kTallRows : kShortRows> {
    using G = Rows<FT, sizeof(FT) == 4 ? kTallRows : kShortRows>;
    static constexpr int B = (int)sizeof(FT);
    static constexpr int DER = G::F32 ? G::LEAD * 8 : 0;
    static constexpr int C = DER + 5 * G::TILE * B + (G::F32 && G::H * 8 > 4 * G::TILE * B ? G::H * 8 : 0);
    static constexpr int LEAD_ = G::F32 ? 0 : C + 4 * G::TILE * B;
    static constexpr int RING = G::F32 ? DER + 9 * G::TILE * B + G::H * 8 : LEAD_ + G::LEAD * 8;
    static constexpr int WZ = RING + 8 * G::HALO * B + (G::F32 ? 0 : G::H * 8), LVA = WZ + G::TILE * B,
                         UXA = LVA + G::LV * B, LUA = UXA + G::LV * B, VYA = LUA + G::LU * B;
};

// 4 bytes a lane from src + off into 256 consecutive bytes of LDS.
__device__ __forceinline__ void dma4(const double *src, unsigned off, void *lds)
{
    asm volatile("" : "+s"(src));  // kept scalar, as in at()
    __builtin_amdgcn_global_load_lds((const void GAS *)((const char GAS *)src + off), (lds_void *)lds, 4, 0, 0);
}

template <typename T>
__device__ __forceinline__ T *uniform(T *p)
{
    const uint64_t a = (uint64_t)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a), hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
    return (T *)((uint64_t)hi << 32 | lo);
}

__device__ __forceinline__ int wrap(int a, int e)
{
    const int r = a % e;
    return r < 0 ? r + e : r;
}

// The arrays of a workgroup in LDS, each an object of its own: reads of one need not wait for
// the DMA into another.
template <typename FT>
struct Shared {
    double *lead, *h;
    FT *c, *der, *lu, *lv, *ux, *vy, *ring, *wz;
    unsigned *lx;
};

// Returns the lane's largest c + |u|, c + |v|, c + |w| of the result (bits; stage 3).
template <typename FT, int STAGE, int ROWS>
__device__ __forceinline__ unsigned long long stage_rows(BoxDev &B, const TileDev &tl, const Shared<FT> &sh)
{
    using KK = K<FT>;
    using L = Lay<FT>;
    using G = Rows<FT, ROWS>;
    constexpr bool F32 = G::F32;
    constexpr int BY = G::BY, R = G::R, NT = G::NT, NW = G::NW, TILE = G::TILE, XH = G::XH, HALO = G::HALO;
    constexpr int LHY = G::LHY, LHX = G::LHX, LU = G::LU, LV = G::LV;
    constexpr int XW = G::XW, YC = G::YC, XC = G::XC, CC = G::CC, VX = G::VX, XS = G::XS;
    double *const s_lead = sh.lead;      // leading plane, raw (cns_stage.hip's layout)
    double *const s_h = sh.h;            // centre plane's halo, raw
    FT *const s_c = sh.c;                // centre plane: mx, my, mz, E
    FT *const der = sh.der;              // centre plane, derived
    FT *const s_lu = sh.lu;              // leading u: own rows, column c (0..39)
    FT *const s_lv = sh.lv;              // leading v: row r (0..R-1), column 4+c
    FT *const s_ux = sh.ux, *const s_vy = sh.vy, *const s_wz = sh.wz;
    FT *const s_ring = sh.ring;          // w of plane p on the halo columns, slot p % 8
    unsigned *const s_lx = sh.lx;        // a lane's column in a staged row of 32 cells
    auto my_tid = []() {  // opaque_tid() of this many threads
        unsigned t = threadIdx.x;
        asm volatile("" : "+v"(t));
        return t & ((1u << (32 - __builtin_clz(NT - 1))) - 1);
    };
    const int x0 = __builtin_amdgcn_readfirstlane(tl.x0), y0 = __builtin_amdgcn_readfirstlane(tl.y0);
    const int kbeg = __builtin_amdgcn_readfirstlane(tl.z0), kend = kbeg + __builtin_amdgcn_readfirstlane(tl.nz);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // (scalars for certain: with two bodies in a kernel the compiler no longer proves it of all)
    const int e = __builtin_amdgcn_readfirstlane(B.e);
    const int64_t e2 = (int64_t)e * e, e3 = e2 * e;
    const double *cons = uniform(STAGE == 1 ? B.U : (STAGE == 2 ? B.S1 : B.S2));
    const double *base = uniform(B.U);
    double *out = uniform(STAGE == 1 ? B.S1 : (STAGE == 2 ? B.S2 : B.U));
    const double dt = B.dt, pref = B.pref;
    const double ra = STAGE == 1 ? 0.0E0 : (STAGE == 2 ? ThreeQuarters : OneThird);
    const double rb = STAGE == 1 ? 1.0E0 : (STAGE == 2 ? OneQuarter : TwoThirds);
    const FT prefF = (FT)pref, eta = (FT)B.eta, alam = (FT)B.alam;
    const FT dxi0 = (FT)B.dxi[0], dxi1 = (FT)B.dxi[1], dxi2 = (FT)B.dxi[2];
    const FT dxi0s = (FT)(B.dxi[0] * B.dxi[0]), dxi1s = (FT)(B.dxi[1] * B.dxi[1]), dxi2s = (FT)(B.dxi[2] * B.dxi[2]);

    auto wv = [&]() {
        int w = wave;
        asm volatile("" : "+s"(w));
        return w;
    };
    // Byte offsets within a plane.  Staging: own rows 2 wave, 2 wave + 1 and halo row `wave` of
    // the tile (scalars; eight waves) with the lane's column; the x halo's slot `wave` or, past
    // those, the corners'.
    unsigned row8[2], hrow8, xh;
    {
        const unsigned tid = threadIdx.x, lane = tid & 63, half = (lane & 1) * 4;
        for (int j = 0; j < 2; j++) row8[j] = (unsigned)(wrap(y0 + 2 * wave + j, e) * e) * 8u;
        const int hw = wave & 7;
        hrow8 = (unsigned)(wrap(y0 - 4 + (hw < 4 ? hw : hw + BY), e) * e) * 8u;
        if (wave == 0) s_lx[lane] = (unsigned)wrap(x0 + (int)(lane >> 1), e) * 8u + half;
        const bool xs = wave < XS;
        const int h = 32 * (xs ? wave : (wave - XS) & 1) + (int)(lane >> 1), c8 = h & 7, c = c8 < 4 ? c8 : c8 + TX;
        const int r = xs ? (h >> 3) + 4 : (h >> 3) + ((h >> 3) < 4 ? 0 : BY);
        xh = (unsigned)(wrap(y0 + r - 4, e) * e + wrap(x0 + c - 4, e)) * 8u + half;
    }
    __syncthreads();
    // the lane's own cell, in the box or clamped to it
    struct Cell {
        bool active;
        unsigned own8;
    };
    auto cell = [&]() {
        const unsigned tid = my_tid();
        const int i = x0 + (int)(tid & (TX - 1)), j = y0 + (int)(tid / TX);
        return Cell{i < e && j < e, (mul24(min(j, e - 1), e) + (unsigned)min(i, e - 1)) * 8u};
    };
    auto issue_centre = [&](int k) {  // halo of centre plane k
        const double *p = cons + k * e2;
        const int w = wv(), yr = w < 4 ? w : w + BY;
        const unsigned lx = s_lx[my_tid() & 63];
        const double *ph = (const double *)((const char *)p + hrow8);
        if (w < 8) {
            dma4(ph, lx, s_h + 32 * w);
#pragma unroll
            for (int f = 1; f < 5; f++) {
                if (F32)
                    dma4(ph + f * e3, lx, s_h + f * YH + 32 * w);
                else
                    dma4(ph + f * e3, lx, s_c + (f - 1) * TILE + yr * PX + 4);
            }
        }
        if (w < XS) {
#pragma unroll
            for (int f = 0; f < 5; f++) dma4(p + f * e3, xh, s_h + G::HX + f * XH + 32 * w);
        } else if (w < XS + 2) {
#pragma unroll
            for (int f = 0; f < 3; f++) dma4(p + f * e3, xh, s_h + G::HC + f * CORN + 32 * (w - XS));
        }
    };
    auto issue_lead = [&](int k) {  // leading plane of centre plane k
        const int kl = k + 4;
        const double *p = cons + (kl >= e ? kl - e : kl) * e2;  // k + 4 < 2 e
        const int w = wv();
        const unsigned lx = s_lx[my_tid() & 63];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const double *pr = (const double *)((const char *)p + row8[j]);
#pragma unroll
            for (int f = 0; f < 5; f++) dma4(pr + f * e3, lx, s_lead + f * NT + (2 * w + j) * TX);
        }
        const double *ph = (const double *)((const char *)p + hrow8);
        if (w < 8) {
            dma4(ph, lx, s_lead + LHY + 32 * w);
            dma4(ph + IMY * e3, lx, s_lead + LHY + YH + 32 * w);
            dma4(ph + IMZ * e3, lx, s_lead + LHY + 2 * YH + 32 * w);
        }
        if (w < XS) {
            dma4(p, xh, s_lead + LHX + 32 * w);
            dma4(p + IMX * e3, xh, s_lead + LHX + XH + 32 * w);
            dma4(p + IMZ * e3, xh, s_lead + LHX + 2 * XH + 32 * w);
        }
    };

    // Windows: plane k+m of the own column at [4+m].  FP64 keeps 1/rho and forms u, v, w as one
    // product; FP32 keeps them rounded.
    FT wmx[9], wmy[9], wmz[9], wE[9], wp[9], wT[9], wux[9], wvy[9], wu[9], wv_[9], ww[9];
    double wri[9];
#define WU(m) (F32 ? wu[m] : (FT)(wmx[m] * wri[m]))
#define WV(m) (F32 ? wv_[m] : (FT)(wmy[m] * wri[m]))
#define WW(m) (F32 ? ww[m] : (FT)(wmz[m] * wri[m]))
    // primitives of a cell into window entry m; gives u, v
    auto window = [&](int m, double r, double mx, double my, double mz, double E, FT &u, FT &v) {
        double u_, v_, w_, eint, p_;
        ctoprim_cell(r, mx, my, mz, E, u_, v_, w_, eint, p_);
        wmx[m] = (FT)mx;
        wmy[m] = (FT)my;
        wmz[m] = (FT)mz;
        wE[m] = (FT)E;
        u = (FT)u_;
        v = (FT)v_;
        if (F32) {
            wu[m] = u;
            wv_[m] = v;
            ww[m] = (FT)w_;
            wp[m] = (FT)(p_ - pref);
            wT[m] = (FT)(eint / CV);
            pin(wu[m], wv_[m], ww[m], wp[m], wT[m], wmx[m], wmy[m], wmz[m], wE[m]);
        } else {
            wri[m] = 1.0E0 / r;
            wp[m] = (FT)p_;
            wT[m] = (FT)(eint / CV);
            pin(wri[m], wp[m], wT[m]);
        }
    };
    auto shift = [&]() {
#pragma unroll
        for (int m = 0; m < 8; m++) {
            wmx[m] = wmx[m + 1]; wmy[m] = wmy[m + 1]; wmz[m] = wmz[m + 1]; wE[m] = wE[m + 1];
            wp[m] = wp[m + 1]; wT[m] = wT[m + 1]; wux[m] = wux[m + 1]; wvy[m] = wvy[m + 1];
            if (F32) {
                wu[m] = wu[m + 1]; wv_[m] = wv_[m + 1]; ww[m] = ww[m + 1];
            } else {
                wri[m] = wri[m + 1];
            }
        }
    };

    // primitives of the leading plane: own cell into the windows' entry 8, u and v with their
    // halos into the lead tiles, w of the halo columns
    auto lead = [&]() {
        const unsigned tid = my_tid(), col = tid & (TX - 1), row = tid / TX;
        FT u, v;
        window(8, s_lead[tid], s_lead[RMX * NT + tid], s_lead[RMY * NT + tid], s_lead[RMZ * NT + tid],
               s_lead[RE * NT + tid], u, v);
        s_lu[mul24(row, PX) + col + 4] = u;
        s_lv[(row + 4) * TX + col] = v;
        const int w = wv();
        if (w < 4) {
            const unsigned yr = row < 4 ? row : row + BY;  // waves 0..3: rows 0..7
            const double hinv = 1.0E0 / s_lead[LHY + tid];
            s_lv[yr * TX + col] = (FT)(s_lead[LHY + YH + tid] * hinv);
            s_wz[mul24(yr, PX) + col + 4] = (FT)(s_lead[LHY + 2 * YH + tid] * hinv);
        }
        if (w >= 4 && w < 4 + XW) {
            const unsigned xid = tid - 256, c8 = xid & 7;
            const double hinv = 1.0E0 / s_lead[LHX + xid];
            const unsigned l = mul24(xid >> 3, PX) + (c8 < 4 ? c8 : c8 + TX);
            s_lu[l] = (FT)(s_lead[LHX + XH + xid] * hinv);
            s_wz[l + 4 * PX] = (FT)(s_lead[LHX + 2 * XH + xid] * hinv);
        }
    };

    // ux, vy of the leading plane into the windows; wz on the halo columns (cns_stage.hip)
    auto lead_grads = [&](int k) {
        const unsigned tid = my_tid(), col = tid & (TX - 1), row = tid / TX;
        FT a[9], b[9];
        {
            const Taps<L::LUA, FT> p_lu(s_lu, mul24(row, PX) + col);
            const Taps<L::LVA, FT> p_lv(s_lv, tid);
#pragma unroll
            for (int m = 0; m < 9; m++)
                if (m != 4) {
                    a[m] = p_lu[m];
                    b[m] = p_lv[m * TX];
                }
            FENCE();
        }
#define GA(mm) a[4 + (mm)]
#define GB(mm) b[4 + (mm)]
        wux[8] = KD1(GA) * dxi0;
        wvy[8] = KD1(GB) * dxi1;
        pin(wux[8], wvy[8]);
        FENCE();
        const int w = wv();
        if (w < 4 + XW) {
            const unsigned xid = tid - 256, c8 = xid & 7;
            const unsigned rc = w < 4 ? tid : YH + xid;
            const unsigned l = w < 4 ? mul24(row < 4 ? row : row + BY, PX) + col + 4
                               : mul24((xid >> 3) + 4, PX) + (c8 < 4 ? c8 : c8 + TX);
            const Taps<0, FT> p_r(s_ring, rc);
            a[8] = s_wz[l];  // w of plane k+4, left here by lead()
#pragma unroll
            for (int m = 0; m < 8; m++)
                if (m != 4) a[m] = p_r[((k + m) & 7) * HALO];
            FENCE();
            s_wz[l] = KD1(GA) * dxi2;
            s_ring[(k & 7) * HALO + rc] = a[8];
        }
    };

    // Fill the windows and the ring with planes kbeg-4 .. kbeg+3, all at once (cns_stage.hip)
    {
        FT *const fl = (FT *)s_lead;
        FT *const lu[8] = {fl, fl + LU, fl + 2 * LU, fl + 3 * LU, s_lu, s_ux, s_vy, s_wz};
        FT *const lv[8] = {fl + 4 * LU, s_lv, der, der + LV, der + 2 * LV, der + 3 * LV, der + 4 * LV, der + 5 * LV};
        const unsigned tid = my_tid(), col = tid & (TX - 1), row = tid / TX;
        const unsigned xid = tid - 256, c8 = xid & 7, xcol = c8 < 4 ? c8 : c8 + TX, yrow = row < 4 ? row : row + BY;
        const bool yl = wave < 4, halo = wave < 4 + XW;
        double cr[8], cx[8], cy[8], cz[8], cE[8], hr[8], hm[8], hz[8];
        {
            const int hy = yl ? (int)yrow : (int)(xid >> 3) + 4, hx = yl ? (int)col + 4 : (int)xcol;
            const unsigned h8 = (unsigned)(wrap(y0 + hy - 4, e) * e + wrap(x0 + hx - 4, e)) * 8u;
            const unsigned own8 = (unsigned)(wrap(y0 + (int)row, e) * e + wrap(x0 + (int)col, e)) * 8u;
#pragma unroll
            for (int m = 0; m < 8; m++) {
                const double *p = cons + wrap(kbeg - 4 + m, e) * e2;
                cr[m] = at(p, own8);
                cx[m] = at(p + IMX * e3, own8);
                cy[m] = at(p + IMY * e3, own8);
                cz[m] = at(p + IMZ * e3, own8);
                cE[m] = at(p + IENE * e3, own8);
                hr[m] = hm[m] = hz[m] = 1.0;
                if (halo) {
                    hr[m] = at(p, h8);
                    hm[m] = at(p + (yl ? IMY : IMX) * e3, h8);
                    hz[m] = at(p + IMZ * e3, h8);
                }
            }
        }
        issue_centre(kbeg);
        FENCE();
#pragma unroll
        for (int m = 0; m < 8; m++) {
            FT u, v;
            window(m, cr[m], cx[m], cy[m], cz[m], cE[m], u, v);
            lu[m][mul24(row, PX) + col + 4] = u;
            lv[m][(row + 4) * TX + col] = v;
            if (halo) {
                const double hinv = 1.0E0 / hr[m];
                if (yl)
                    lv[m][yrow * TX + col] = (FT)(hm[m] * hinv);
                else
                    lu[m][mul24(xid >> 3, PX) + xcol] = (FT)(hm[m] * hinv);
                s_ring[((kbeg + m) & 7) * HALO + (yl ? tid : YH + xid)] = (FT)(hz[m] * hinv);
            }
            FENCE();
        }
        __syncthreads();
        auto grads = [&](int m) {
            lds_tap<FT> *p_lu = (lds_tap<FT> *)lu[m] + mul24(row, PX) + col, *p_lv = (lds_tap<FT> *)lv[m] + tid;
            FT a[9], b[9];
#pragma unroll
            for (int i = 0; i < 9; i++)
                if (i != 4) {
                    a[i] = p_lu[i];
                    b[i] = p_lv[i * TX];
                }
            wux[m] = KD1(GA) * dxi0;
            wvy[m] = KD1(GB) * dxi1;
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

    unsigned long long cmax = 0ull;  // bits of max(c + |u|, c + |v|, c + |w|)
#pragma unroll 1
    for (int k = kbeg; k < kend; k++) {
        const FT *d_u = der + VU * TILE, *d_v = der + VV * TILE;
        // ---------------- phase 1: primitives of the leading plane, tiles of the centre plane
        lead();
        {
            const unsigned tid = my_tid(), col = tid & (TX - 1), row = tid / TX, lane = tid & 63;
            const unsigned me = mul24(row + 4, PX) + col + 4;
            der[VU * TILE + me] = WU(4);
            der[VV * TILE + me] = WV(4);
            der[VW * TILE + me] = WW(4);
            der[VT * TILE + me] = wT[4];
            der[VP * TILE + me] = wp[4];
            s_c[me] = wmx[4];
            s_c[TILE + me] = wmy[4];
            s_c[2 * TILE + me] = wmz[4];
            s_c[3 * TILE + me] = wE[4];
            auto halo_prim = [&](unsigned l, double r, double mx, double my, double mz, double E) {
                double u_, v_, w_, eint, p_;
                ctoprim_cell(r, mx, my, mz, E, u_, v_, w_, eint, p_);
                der[VU * TILE + l] = (FT)u_;
                der[VV * TILE + l] = (FT)v_;
                der[VW * TILE + l] = (FT)w_;
                der[VT * TILE + l] = (FT)(eint / CV);
                der[VP * TILE + l] = F32 ? (FT)(p_ - pref) : (FT)p_;
            };
            auto halo_cons = [&](unsigned l, double mx, double my, double mz, double E) {
                s_c[l] = (FT)mx;
                s_c[TILE + l] = (FT)my;
                s_c[2 * TILE + l] = (FT)mz;
                s_c[3 * TILE + l] = (FT)E;
            };
            const int w = wv();
            if (w >= YC) {
                const unsigned yrow = row - 2 * YC, l = mul24(yrow < 4 ? yrow : yrow + BY, PX) + col + 4, h = tid - 64 * YC;
                if (F32) {
                    const double mx = s_h[YH + h], my = s_h[2 * YH + h], mz = s_h[3 * YH + h], E = s_h[4 * YH + h];
                    halo_cons(l, mx, my, mz, E);
                    halo_prim(l, s_h[h], mx, my, mz, E);
                } else {
                    halo_prim(l, s_h[h], s_c[l], s_c[TILE + l], s_c[2 * TILE + l], s_c[3 * TILE + l]);
                }
            }
            if (w >= XC && w < XC + XW) {
                const unsigned xid = tid - 64 * XC, c8 = xid & 7, l = mul24((xid >> 3) + 4, PX) + (c8 < 4 ? c8 : c8 + TX);
                const double *h = s_h + G::HX + xid;
                const double mx = h[XH], my = h[2 * XH], mz = h[3 * XH], E = h[4 * XH];
                halo_cons(l, mx, my, mz, E);
                halo_prim(l, h[0], mx, my, mz, E);
            }
            if (w == CC) {  // u and v only
                const unsigned r8 = lane >> 3, c8 = lane & 7;
                const unsigned l = mul24(r8 < 4 ? r8 : r8 + BY, PX) + (c8 < 4 ? c8 : c8 + TX);
                const double *h = s_h + G::HC;
                const double cinv = 1.0E0 / h[lane];
                der[VU * TILE + l] = (FT)(h[CORN + lane] * cinv);
                der[VV * TILE + l] = (FT)(h[2 * CORN + lane] * cinv);
            }
        }
        __syncthreads();  // B

        // ---------------- phase 2
        // Of the two waves of a SIMD the older wins every choice, and would wait at C while the
        // younger (4..7) runs alone: the younger goes first up to the end of the z terms.
        if (wave >= 8)
            __builtin_amdgcn_s_setprio(2);
        else if (wave >= 4)
            __builtin_amdgcn_s_setprio(1);
        if (k + 1 < kend) issue_lead(k + 1);
        FT F[5], zf[5];
        lead_grads(k);
        {
            const unsigned tid = my_tid(), col = tid & (TX - 1), row = tid / TX;
            // ux, vy of the centre plane: own cells from the windows, the halos the mixed
            // derivatives read from the derived tiles (cpu/diffterm.cpp:77-151)
            s_ux[(row + 4) * TX + col] = wux[4];
            const int w = wv();
            FT a[9];
            if (w >= YC) {
                const unsigned yrow = row - 2 * YC, yr = yrow < 4 ? yrow : yrow + BY;
                const Taps<L::DER, FT> p_u(d_u, mul24(yr, PX) + col);
#pragma unroll
                for (int m = 0; m < 9; m++)
                    if (m != 4) a[m] = p_u[m];
                FENCE();
                s_ux[yr * TX + col] = KD1(GA) * dxi0;
            }
            s_vy[mul24(row, PX) + col + 4] = wvy[4];
            if (w >= VX && w < VX + XW) {
                const unsigned xid = tid - 64 * VX, c8 = xid & 7, l = mul24(xid >> 3, PX) + (c8 < 4 ? c8 : c8 + TX);
                const Taps<L::DER, FT> p_v(d_v, l);
#pragma unroll
                for (int m = 0; m < 9; m++)
                    if (m != 4) a[m] = p_v[m * PX];
                FENCE();
                s_vy[l] = KD1(GA) * dxi1;
            }
            FENCE();
        }
#undef GA
#undef GB
        FT zx = 0, zy = 0, zz = 0, zt = 0, uz = 0, vz = 0, mz = 0;
        {
            // every z term of the cell, from the windows
            FT hs[5], uxz, vyz, wzc;
            zx = KK::CENTER * WU(4);
            zy = KK::CENTER * WV(4);
            zz = KK::CENTER * WW(4);
            zt = KK::CENTER * wT[4];
#define ZTAP(m, C1, C2, FIRST)                                                                                   \
    {                                                                                                            \
        const FT w1 = WW(4 + m), w0 = WW(4 - m), q1 = F32 ? wp[4 + m] + prefF : wp[4 + m],                       \
                 q0 = F32 ? wp[4 - m] + prefF : wp[4 - m];                                                       \
        hyp_tap<FIRST>(C1, wmz[4 + m], wmz[4 - m], wmx[4 + m], wmx[4 - m], wmy[4 + m], wmy[4 - m], wE[4 + m],     \
                       wE[4 - m], wp[4 + m], wp[4 - m], q1, q0, w1, w0, hs);                                     \
        tap<FIRST>(wzc, C1 * (w1 - w0));                                                                         \
        tap<false>(zz, C2 * (w1 + w0));                                                                          \
        const FT u1 = WU(4 + m), u0 = WU(4 - m);                                                                 \
        tap<FIRST>(uz, C1 * (u1 - u0));                                                                          \
        tap<false>(zx, C2 * (u1 + u0));                                                                          \
        const FT v1 = WV(4 + m), v0 = WV(4 - m);                                                                 \
        tap<FIRST>(vz, C1 * (v1 - v0));                                                                          \
        tap<false>(zy, C2 * (v1 + v0));                                                                          \
        tap<false>(zt, C2 * (wT[4 + m] + wT[4 - m]));                                                            \
        tap<FIRST>(uxz, C1 * (wux[4 + m] - wux[4 - m]));                                                         \
        tap<FIRST>(vyz, C1 * (wvy[4 + m] - wvy[4 - m]));                                                         \
        pin(hs[0], hs[1], hs[2], hs[3], hs[4], wzc, zz, uz, zx, vz, zy, zt, uxz, vyz);                            \
        FENCE();                                                                                                 \
    }
            ZTAP(1, KK::ALP, KK::OFF1, true)
            ZTAP(2, KK::BET, KK::OFF2, false)
            ZTAP(3, KK::GAM, KK::OFF3, false)
            ZTAP(4, KK::DEL, KK::OFF4, false)
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
            const unsigned tid = my_tid();
            s_wz[mul24(tid / TX + 4, PX) + (tid & (TX - 1)) + 4] = wzc;
        }
        __builtin_amdgcn_s_setprio(0);
        shift();  // the centre plane is window entry 3 from here
        constexpr int Z = 4 * PX;
        {
            // from four rows above the own cell: every tap is a non-negative constant away
            const unsigned tid = my_tid(), me4 = mul24(tid / TX, PX) + (tid & (TX - 1)) + 4;
            const Taps<L::C, FT> s_m(s_c, me4);
            const Taps<L::DER, FT> s_d(der, me4);
            FT hs[5], A[12];
            enum { CX = 0, CY, CZ, CE };
            // fields n, a, b, E of the conserved tile, p and v of the derived one at taps +o and -o
            auto load = [&](FT (&T)[12], int n, int a_, int b_, int v, int o) {
                T[0] = s_m[n * TILE + Z + o]; T[1] = s_m[n * TILE + Z - o];
                T[2] = s_m[a_ * TILE + Z + o]; T[3] = s_m[a_ * TILE + Z - o];
                T[4] = s_m[b_ * TILE + Z + o]; T[5] = s_m[b_ * TILE + Z - o];
                T[6] = s_m[CE * TILE + Z + o]; T[7] = s_m[CE * TILE + Z - o];
                T[8] = s_d[VP * TILE + Z + o]; T[9] = s_d[VP * TILE + Z - o];
                T[10] = s_d[v * TILE + Z + o]; T[11] = s_d[v * TILE + Z - o];
            };
#define HT(FIRST, C, T)                                                                                    \
    {                                                                                                      \
        const FT q1 = F32 ? T[8] + prefF : T[8], q0 = F32 ? T[9] + prefF : T[9];                           \
        hyp_tap<FIRST>(C, T[0], T[1], T[2], T[3], T[4], T[5], T[6], T[7], T[8], T[9], q1, q0, T[10], T[11], hs); \
        pin(hs[0], hs[1], hs[2], hs[3], hs[4]);                                                            \
        FENCE();                                                                                           \
    }
            load(A, CX, CY, CZ, VU, 1); FENCE();
            HT(true, KK::ALP, A)
            load(A, CX, CY, CZ, VU, 2); FENCE();
            HT(false, KK::BET, A)
            load(A, CX, CY, CZ, VU, 3); FENCE();
            HT(false, KK::GAM, A)
            load(A, CX, CY, CZ, VU, 4); FENCE();
            HT(false, KK::DEL, A)
            F[IRHO] = -(hs[0]) * dxi0;
            F[IMX] = -(hs[1]) * dxi0;
            F[IMY] = -(hs[2]) * dxi0;
            F[IMZ] = -(hs[3]) * dxi0;
            F[IENE] = -(hs[4]) * dxi0;
            load(A, CY, CX, CZ, VV, PX); FENCE();
            HT(true, KK::ALP, A)
            load(A, CY, CX, CZ, VV, 2 * PX); FENCE();
            HT(false, KK::BET, A)
            load(A, CY, CX, CZ, VV, 3 * PX); FENCE();
            HT(false, KK::GAM, A)
            load(A, CY, CX, CZ, VV, 4 * PX); FENCE();
            HT(false, KK::DEL, A)
#undef HT
            F[IRHO] = F[IRHO] - hs[0] * dxi1;
            F[IMY] = F[IMY] - hs[1] * dxi1;
            F[IMX] = F[IMX] - hs[2] * dxi1;
            F[IMZ] = F[IMZ] - hs[3] * dxi1;
            F[IENE] = F[IENE] - hs[4] * dxi1;
#pragma unroll
            for (int l = 0; l < NC; l++) F[l] = F[l] - zf[l];
            pin(F[0], F[1], F[2], F[3], F[4]);
        }
        __syncthreads();  // C

        // ---------------- phase 3
        if (k + 1 < kend) issue_centre(k + 1);
        {   // held in the lead tile's own cells (read by the neighbours before C) until the update
            const unsigned tid = my_tid(), col = tid & (TX - 1), row = tid / TX;
            s_lv[(row + 4) * TX + col] = F[IENE];
        }
        {
            // diffterm's x and y terms, from the tiles, then its sums (cpu/diffterm.cpp:159-311)
            const unsigned tid = my_tid(), col = tid & (TX - 1), row = tid / TX;
            const unsigned me4 = mul24(row, PX) + col + 4;
            const Taps<L::DER, FT> s_d(der, me4);
            const Taps<L::WZ, FT> s_z(s_wz, me4);
            const Taps<L::VYA, FT> s_m4(s_vy, me4 - 4);
            FT A[12], xu, xv, xw, xt, d2v, d2w, m1, m2;
            // u, v, w, T of the derived tile, wz and vy at taps +o and -o in x
            auto load = [&](FT (&T)[12], int o) {
                T[0] = s_d[VU * TILE + Z + o]; T[1] = s_d[VU * TILE + Z - o];
                T[2] = s_d[VV * TILE + Z + o]; T[3] = s_d[VV * TILE + Z - o];
                T[4] = s_d[VW * TILE + Z + o]; T[5] = s_d[VW * TILE + Z - o];
                T[6] = s_d[VT * TILE + Z + o]; T[7] = s_d[VT * TILE + Z - o];
                T[8] = s_z[Z + o]; T[9] = s_z[Z - o];
                T[10] = s_m4[4 + o]; T[11] = s_m4[4 - o];
            };
            // second differences of u, v, w, T; first of v (d2v), w (d2w), and of the two mixed terms
#define DT(FIRST, C1, C2, T)                     \
    tap<false>(xu, C2 * (T[0] + T[1]));          \
    tap<false>(xv, C2 * (T[2] + T[3]));          \
    tap<false>(xw, C2 * (T[4] + T[5]));          \
    tap<false>(xt, C2 * (T[6] + T[7]));          \
    tap<FIRST>(d2v, C1 * (T[2] - T[3]));         \
    tap<FIRST>(d2w, C1 * (T[4] - T[5]));         \
    tap<FIRST>(m1, C1 * (T[10] - T[11]));        \
    tap<FIRST>(m2, C1 * (T[8] - T[9]));          \
    pin(xu, xv, xw, xt, d2v, d2w, m1, m2);       \
    FENCE()
            xu = KK::CENTER * WU(3);
            xv = KK::CENTER * WV(3);
            xw = KK::CENTER * WW(3);
            xt = KK::CENTER * wT[3];
            load(A, 1); FENCE();
            DT(true, KK::ALP, KK::OFF1, A);
            load(A, 2); FENCE();
            DT(false, KK::BET, KK::OFF2, A);
            load(A, 3); FENCE();
            DT(false, KK::GAM, KK::OFF3, A);
            load(A, 4); FENCE();
            DT(false, KK::DEL, KK::OFF4, A);
#undef DT
            FT sx = KK::FourThirds * (xu * dxi0s), sy = xv * dxi0s, sz = xw * dxi0s, st = xt * dxi0s;
            const FT vx = d2v * dxi0, wx = d2w * dxi0, mx = m1 * dxi0 + m2 * dxi0;
            pin(sx, sy, sz, st);
            // the update's operands of the own cell (cells past the box: a valid one's, unused)
            double rkb[5], uc[5];
            {
                const unsigned own8 = cell().own8;
                const double *pc = cons + k * e2, *pb = base + k * e2;
                uc[IRHO] = at(pc, own8);
                if (F32) {
#pragma unroll
                    for (int l = 1; l < NC; l++) uc[l] = at(pc + l * e3, own8);
                }
                if (STAGE != 1) {
#pragma unroll
                    for (int l = 0; l < NC; l++) rkb[l] = at(pb + l * e3, own8);
                }
            }
            const Taps<L::UXA, FT> s_n(s_ux, tid);
            xu = KK::CENTER * WU(3);
            xv = KK::CENTER * WV(3);
            xw = KK::CENTER * WW(3);
            xt = KK::CENTER * wT[3];
            auto ytap = [&](auto first, FT c1, FT c2, int o, int on) {
                constexpr bool FI = decltype(first)::value;
                {
                    const FT u1 = s_d[VU * TILE + Z + o], u0 = s_d[VU * TILE + Z - o], v1 = s_d[VV * TILE + Z + o],
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
                    const FT t1 = s_d[VT * TILE + Z + o], t0 = s_d[VT * TILE + Z - o], z1 = s_z[Z + o], z0 = s_z[Z - o],
                             n1 = s_n[4 * TX + on], n0 = s_n[4 * TX - on];
                    FENCE();
                    tap<false>(xt, c2 * (t1 + t0));
                    tap<FI>(m1, c1 * (n1 - n0));
                    tap<FI>(m2, c1 * (z1 - z0));
                    pin(xt, m1, m2);
                    FENCE();
                }
            };
            ytap(std::true_type(), KK::ALP, KK::OFF1, PX, TX);
            ytap(std::false_type(), KK::BET, KK::OFF2, 2 * PX, 2 * TX);
            ytap(std::false_type(), KK::GAM, KK::OFF3, 3 * PX, 3 * TX);
            ytap(std::false_type(), KK::DEL, KK::OFF4, 4 * PX, 4 * TX);
            sx = sx + xu * dxi1s;
            sy = sy + KK::FourThirds * (xv * dxi1s);
            sz = sz + xw * dxi1s;
            st = st + xt * dxi1s;
            const FT tauxy = d2v * dxi1 + vx, wy = d2w * dxi1, my = m1 * dxi1 + m2 * dxi1;
            const FT uzz = zx, vzz = zy, wzz = zz, tzz = zt;
            FT D[5];
            D[IMX] = eta * (sx + uzz + KK::OneThird * mx);
            D[IMY] = eta * (sy + vzz + KK::OneThird * my);
            D[IMZ] = eta * (sz + KK::FourThirds * wzz + KK::OneThird * mz);
            {
                const FT ux = wux[3], vy = wvy[3], wz = s_z[Z];
                const FT divu = KK::TwoThirds * (ux + vy + wz);
                const FT tauxx = KK::Two * ux - divu;
                const FT tauyy = KK::Two * vy - divu;
                const FT tauzz = KK::Two * wz - divu;
                const FT tauxz = uz + wx;
                const FT tauyz = vz + wy;
                FT mechwork = tauxx * ux + tauyy * vy + tauzz * wz + (tauxy * tauxy) + (tauxz * tauxz)
                              + (tauyz * tauyz);
                mechwork = eta * mechwork + D[IMX] * WU(3) + D[IMY] * WV(3) + D[IMZ] * WW(3);
                D[IENE] = alam * (st + tzz) + mechwork;
            }
            F[IENE] = s_lv[(row + 4) * TX + col];
            if (!F32) {
                uc[IMX] = wmx[3];
                uc[IMY] = wmy[3];
                uc[IMZ] = wmz[3];
                uc[IENE] = wE[3];
            }
            // the next plane's halo has landed before the stores join the queue, so the barrier
            // that ends the phase need not wait for them
            __builtin_amdgcn_s_waitcnt(0xF70);
            const Cell c = cell();
            if (c.active) {
                const unsigned own8 = c.own8;
                double o[5];
#pragma unroll
                for (int l = 0; l < NC; l++) {
                    // cpu/advance.cpp:82, :114-116, :148-150
                    const double df = (l == 0 ? 0.0E0 : (double)D[l]) + (double)F[l];
                    const double x = uc[l] + dt * df;
                    o[l] = STAGE == 1 ? x : ra * rkb[l] + rb * x;
                    at(out + k * e2 + l * e3, own8) = o[l];
                }
                if (STAGE == 3) {
                    // (c + |u|) / dx of the three directions, cpu/ctoprim.cpp:52-59.  A box's dx is
                    // the same in all three, and rounded division by it keeps order: the largest
                    // quotient is that of the largest sum, divided once a tile instead of per cell.
                    double u, v, w, eint, p;
                    ctoprim_cell(o[IRHO], o[IMX], o[IMY], o[IMZ], o[IENE], u, v, w, eint, p);
                    const double cs = sqrt(GAMMA * p / o[IRHO]);
                    const unsigned long long b0 = courno_bits(cs + fabs(u)), b1 = courno_bits(cs + fabs(v)),
                                             b2 = courno_bits(cs + fabs(w));
                    cmax = cmax > b0 ? cmax : b0;
                    cmax = cmax > b1 ? cmax : b1;
                    cmax = cmax > b2 ? cmax : b2;
                }
            }
        }
        __syncthreads();  // A
    }
#undef WU
#undef WV
#undef WW
    return cmax;
}

template <typename FT, int STAGE>
__global__ void __launch_bounds__(Lay<FT>::NT, Lay<FT>::NW / 4)
batch_stage_kernel(BoxDev *__restrict__ boxes, const TileDev *__restrict__ tiles, int ntiles)
{
    using L = Lay<FT>;
    __shared__ double s_lead[L::LEAD];
    __shared__ double s_h[L::H];
    __shared__ FT s_c[4 * L::TILE];
    __shared__ FT der[VNF * L::TILE];
    __shared__ FT s_lu[L::LU];
    __shared__ FT s_lv[L::LV];
    __shared__ FT s_ux[L::LV];
    __shared__ FT s_vy[L::LU];
    __shared__ FT s_ring[8 * L::HALO];
    __shared__ FT s_wz[L::TILE];
    __shared__ unsigned s_lx[64];
    __shared__ unsigned long long s_red[L::NW];

    const int ti = xcd_tile(blockIdx.x, gridDim.x);
    if (ti >= ntiles) return;
    const TileDev tl = tiles[ti];
    if (tl.nz == 0) return;  // filler of an XCD's part of the list
    BoxDev &B = boxes[__builtin_amdgcn_readfirstlane(tl.box)];
    if (box_stopped(B)) return;  // uniform over the workgroup
    const Shared<FT> sh{s_lead, s_h, s_c, der, s_lu, s_lv, s_ux, s_vy, s_ring, s_wz, s_lx};
    const int rows = L::F32 ? __builtin_amdgcn_readfirstlane(tl.rows) : kShortRows, waves = rows / 2;
    unsigned long long cmax;
    if (L::F32 && rows == kTallRows) {
        cmax = stage_rows<FT, STAGE, L::BY>(B, tl, sh);
    } else {
        // (a wave that has ended no longer counts at the barriers)
        if (__builtin_amdgcn_readfirstlane(threadIdx.x) >= TX * kShortRows) return;
        cmax = stage_rows<FT, STAGE, kShortRows>(B, tl, sh);
    }
    if (STAGE == 3) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const unsigned long long v = __shfl_xor(cmax, off);
            cmax = cmax > v ? cmax : v;
        }
        if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = cmax;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 0; w < waves; w++) cmax = cmax > s_red[w] ? cmax : s_red[w];
            atomicMax(&B.acc, courno_bits(__longlong_as_double((long long)cmax) / B.dx[0]));
        }
    }
}

}  // namespace

hipError_t launch_batch_fused(BoxDev *boxes, const TileDev *tiles, int n, int stage, bool fp32, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
#define BATCH_STAGE(FT)                                                               \
    switch (stage) {                                                                  \
    case 1: batch_stage_kernel<FT, 1><<<n, Lay<FT>::NT, 0, s>>>(boxes, tiles, n); break; \
    case 2: batch_stage_kernel<FT, 2><<<n, Lay<FT>::NT, 0, s>>>(boxes, tiles, n); break; \
    case 3: batch_stage_kernel<FT, 3><<<n, Lay<FT>::NT, 0, s>>>(boxes, tiles, n); break; \
    default: return hipErrorInvalidValue;                                             \
    }
    if (fp32) {
        BATCH_STAGE(float)
    } else {
        BATCH_STAGE(double)
    }
#undef BATCH_STAGE
    return hipGetLastError();
}

}  // namespace cns
