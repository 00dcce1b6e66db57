// cns_pipe_tile.h -- pieces shared by the z-marching, DMA-staged stencil kernels (internal):
// difference sums, the XCD-aware tile order, direct-to-LDS loads of a haloed tile, hypterm's
// flux of a cell and the stage update with its stores.
#pragma once

#include "cns_kernels.h"

namespace cns {

namespace {

typedef __attribute__((address_space(3))) void lds_void;

#define D1(F) (ALP * (F(1) - F(-1)) + BET * (F(2) - F(-2)) + GAM * (F(3) - F(-3)) + DEL * (F(4) - F(-4)))
#define D2(F)                                                                                \
    (CENTER * F(0) + OFF1 * (F(1) + F(-1)) + OFF2 * (F(2) + F(-2)) + OFF3 * (F(3) + F(-3)) \
     + OFF4 * (F(4) + F(-4)))
#define HMOM(C, UN) \
    (ALP * (C(1) * UN(1) - C(-1) * UN(-1)) + BET * (C(2) * UN(2) - C(-2) * UN(-2)) \
     + GAM * (C(3) * UN(3) - C(-3) * UN(-3)) + DEL * (C(4) * UN(4) - C(-4) * UN(-4)))
#define HMOMP(C, UN, P)                                                                  \
    (ALP * (C(1) * UN(1) - C(-1) * UN(-1) + (P(1) - P(-1)))                              \
     + BET * (C(2) * UN(2) - C(-2) * UN(-2) + (P(2) - P(-2)))                            \
     + GAM * (C(3) * UN(3) - C(-3) * UN(-3) + (P(3) - P(-3)))                            \
     + DEL * (C(4) * UN(4) - C(-4) * UN(-4) + (P(4) - P(-4))))
#define HENE(C, UN, P)                                                                   \
    (ALP * (C(1) * UN(1) - C(-1) * UN(-1) + (P(1) * UN(1) - P(-1) * UN(-1)))             \
     + BET * (C(2) * UN(2) - C(-2) * UN(-2) + (P(2) * UN(2) - P(-2) * UN(-2)))           \
     + GAM * (C(3) * UN(3) - C(-3) * UN(-3) + (P(3) * UN(3) - P(-3) * UN(-3)))           \
     + DEL * (C(4) * UN(4) - C(-4) * UN(-4) + (P(4) * UN(4) - P(-4) * UN(-4))))

__device__ __forceinline__ int xcd_tile(int b, int nb)
{
    const int xcd = b & 7, local = b >> 3;
    const int per = nb >> 3, rem = nb & 7;
    return xcd < rem ? xcd * (per + 1) + local : rem * (per + 1) + (xcd - rem) * per + local;
}

// Tile geometry shared by the DMA issue: the ghosted-array coordinates of tile cell
// (0, 0) and the clamps that keep every lane's 16-byte load inside the array (cells
// beyond the box are only read by lanes whose outputs are discarded).
struct TileDma {
    int gi0, gj0, g1m1, xgm2;
    unsigned xg;
};

// All of this wave's loads, DMA included, have landed; then the workgroup barrier.
__device__ __forceinline__ void plane_barrier()
{
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
}

// Tile shapes of the pipelined stencils: TXs x 8 cells per workgroup of TXs*8
// threads.  At 64 x 8 diffterm takes 142 KB of LDS (one workgroup per CU); at 32 x 8
// 77 KB, so two workgroups share a CU and one's barrier waits are the other's compute
// time (likewise the fused hypterm: 117 KB and 65 KB).
template <int TXs>
struct Shape {
    static constexpr int TX = TXs, BY = 8, PX = TX + 8, R = BY + 8, NT = TX * BY, NW = NT / 64;
    static constexpr int TILE = R * PX, NDMA = TILE / 128;
    static_assert(TILE % 128 == 0, "a tile is a whole number of 1 KB DMA blocks");
    static_assert(PX % 2 == 0, "a lane's 16-byte pair stays in one row");
};

// DMA block n of one field tile: lane L moves tile elements e, e+1 with e = 128 n + 2 L
// (row e / PX, column e % PX; PX is even, so a pair never straddles rows) from the
// plane at `src` into tile + 128 n + 2 L.  A plane offset fits 32 bits; keeping it
// 32-bit halves what the compiler holds live across the plane loop.
template <class S>
__device__ __forceinline__ void dma_block_s(const double *src, double *tile, int n, const TileDma &t, int lane)
{
    const int e = 128 * n + 2 * lane;
    const int r = e / S::PX, c = e - r * S::PX;
    const int hj = min(t.gj0 + r, t.g1m1), hi = min(t.gi0 + c, t.xgm2);
    const unsigned off = (unsigned)hj * t.xg + (unsigned)hi;
    __builtin_amdgcn_global_load_lds((const void *)(src + off), (lds_void *)(tile + 128 * n), 16, 0, 0);
}

// This wave's share of the NF x NDMA DMA blocks of one plane: block n of field f goes
// to wave (n + f) mod NW (NW waves; the last NDMA - NW blocks to the waves after them).
template <class S, int NF>
__device__ __forceinline__ void dma_plane_s(const double *const (&src)[NF], int64_t plane, double *buf,
                                            const TileDma &t, int wave, int lane)
{
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const int n0 = (wave - f) & (S::NW - 1);
        dma_block_s<S>(src[f] + plane, buf + f * S::TILE, n0, t, lane);
        if (n0 + S::NW < S::NDMA) dma_block_s<S>(src[f] + plane, buf + f * S::TILE, n0 + S::NW, t, lane);
    }
}

// hypterm's flux of the lane's cell (LDS index me of 16 x P tiles): x terms from the
// row, y terms from the column, z terms from the register windows (plane k+m at
// [4+m]), in the reference's order (cpu/hypterm.cpp:33-90, :101-147, :158-204).
template <int P>
__device__ __forceinline__ void hyp_flux(const double *s_mx, const double *s_my, const double *s_mz,
                                         const double *s_E, const double *s_p, const double *s_u,
                                         const double *s_v, int me, const double (&wmx)[9],
                                         const double (&wmy)[9], const double (&wmz)[9],
                                         const double (&wE)[9], const double (&ww)[9],
                                         const double (&wp)[9], double dxi0, double dxi1,
                                         double dxi2, double (&F)[5])
{
    // ---- x: F = -(sum)*dxinv(1)
#define XMX(m) s_mx[me + (m)]
#define XMY(m) s_my[me + (m)]
#define XMZ(m) s_mz[me + (m)]
#define XE(m) s_E[me + (m)]
#define XP(m) s_p[me + (m)]
#define XU(m) s_u[me + (m)]
    F[IRHO] = -(D1(XMX)) * dxi0;
    F[IMX] = -(HMOMP(XMX, XU, XP)) * dxi0;
    F[IMY] = -(HMOM(XMY, XU)) * dxi0;
    F[IMZ] = -(HMOM(XMZ, XU)) * dxi0;
    F[IENE] = -(HENE(XE, XU, XP)) * dxi0;
    // ---- y: F = F - (sum)*dxinv(2)
#define YMX(m) s_mx[me + (m) * P]
#define YMY(m) s_my[me + (m) * P]
#define YMZ(m) s_mz[me + (m) * P]
#define YE(m) s_E[me + (m) * P]
#define YP(m) s_p[me + (m) * P]
#define YV(m) s_v[me + (m) * P]
    F[IRHO] = F[IRHO] - (D1(YMY)) * dxi1;
    F[IMX] = F[IMX] - (HMOM(YMX, YV)) * dxi1;
    F[IMY] = F[IMY] - (HMOMP(YMY, YV, YP)) * dxi1;
    F[IMZ] = F[IMZ] - (HMOM(YMZ, YV)) * dxi1;
    F[IENE] = F[IENE] - (HENE(YE, YV, YP)) * dxi1;
    // ---- z: from the register windows
#define ZMX(m) wmx[4 + (m)]
#define ZMY(m) wmy[4 + (m)]
#define ZMZ(m) wmz[4 + (m)]
#define ZE(m) wE[4 + (m)]
#define ZW(m) ww[4 + (m)]
#define ZP(m) wp[4 + (m)]
    F[IRHO] = F[IRHO] - (D1(ZMZ)) * dxi2;
    F[IMX] = F[IMX] - (HMOM(ZMX, ZW)) * dxi2;
    F[IMY] = F[IMY] - (HMOM(ZMY, ZW)) * dxi2;
    F[IMZ] = F[IMZ] - (HMOMP(ZMZ, ZW, ZP)) * dxi2;
    F[IENE] = F[IENE] - (HENE(ZE, ZW, ZP)) * dxi2;
#undef XMX
#undef XMY
#undef XMZ
#undef XE
#undef XP
#undef XU
#undef YMX
#undef YMY
#undef YMZ
#undef YE
#undef YP
#undef YV
#undef ZMX
#undef ZMY
#undef ZMZ
#undef ZE
#undef ZW
#undef ZP
}

// The stage update of the cell and its stores (STAGE1: cons + dt(D+F), the reference's
// form of cpu/advance.cpp:82; later stages ra*base + rb*(cons + dt(D+F)), which is
// 3/4 base + 1/4(..) and 1/3 base + 2/3(..) of :114-116, :148-150).
template <bool STAGE1, bool WRITE_F>
__device__ __forceinline__ void rk_store(const double (&F)[5], const double (&uc)[5], const double (&rkd)[5],
                                         const double (&rkb)[5], double ra, double rb, double dt,
                                         double *flux, int64_t fo, int64_t c, double *out, int64_t zo,
                                         int64_t cg, double (&o)[5])
{
    if (WRITE_F) {
#pragma unroll
        for (int l = 0; l < NC; l++) flux[l * c + fo] = F[l];
    }
#pragma unroll
    for (int l = 0; l < NC; l++) {
        o[l] = STAGE1 ? uc[l] + dt * (rkd[l] + F[l]) : ra * rkb[l] + rb * (uc[l] + dt * (rkd[l] + F[l]));
        out[l * cg + zo] = o[l];
    }
}

// ctoprim of the stage result o at interior cell zo (cpu/ctoprim.cpp:23-38), stored
// into q: u, v, w and T (QOUT 1: what the next stage's diffterm reads) or every
// component (QOUT 2: the Q the reference leaves after a step).  The ghost cells are
// the periodic fill's, so q over the ghosted box equals ctoprim of the filled result.
template <int QOUT>
__device__ __forceinline__ void q_store(const double (&o)[5], double *q, int64_t zo, int64_t cg)
{
    if (QOUT == 0) return;
    double u, v, w, eint, p;
    ctoprim_cell(o[IRHO], o[IMX], o[IMY], o[IMZ], o[IENE], u, v, w, eint, p);
    if (QOUT == 2) q[QRHO * cg + zo] = o[IRHO];
    q[QU * cg + zo] = u;
    q[QV * cg + zo] = v;
    q[QW * cg + zo] = w;
    if (QOUT == 2) q[QPRES * cg + zo] = p;
    q[QTEMP * cg + zo] = eint / CV;
}

}  // namespace

}  // namespace cns
