// cns_pipe_tile.h -- pieces shared by the z-marching, DMA-staged stencil kernels (internal):
// the difference sum, the XCD-aware tile order and direct-to-LDS loads of a haloed tile.
#pragma once

#include "cns_kernels.h"

namespace cns {

namespace {

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) double lds_double;

#define D1(F) (ALP * (F(1) - F(-1)) + BET * (F(2) - F(-2)) + GAM * (F(3) - F(-3)) + DEL * (F(4) - F(-4)))

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
__device__ __forceinline__ void dma_block_s(const double *src, lds_double *tile, int n, const TileDma &t, int lane)
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
__device__ __forceinline__ void dma_plane_s(const double *const (&src)[NF], int64_t plane, lds_double *buf,
                                            const TileDma &t, int wave, int lane)
{
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const int n0 = (wave - f) & (S::NW - 1);
        dma_block_s<S>(src[f] + plane, buf + f * S::TILE, n0, t, lane);
        if (n0 + S::NW < S::NDMA) dma_block_s<S>(src[f] + plane, buf + f * S::TILE, n0 + S::NW, t, lane);
    }
}

}  // namespace

}  // namespace cns
