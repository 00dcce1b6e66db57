// cns_stage_tile.h -- pieces of the one-kernel RK stages (cns_stage.hip, cns_batch_stage.hip):
// the 32 x 16 tile, LDS taps, and the compiler controls that keep a plane's values in
// registers (internal).
#pragma once

#include "cns_pipe_tile.h"

namespace cns {

namespace {

// Tile geometry; sizes are in doubles unless they say otherwise.
constexpr int TX = 32, BY = 16, PX = TX + 8, R = BY + 8, NT = TX * BY, NW = NT / 64;
constexpr int TILE = R * PX;             // a haloed plane
constexpr int YH = 8 * TX, XH = 8 * BY;  // y-halo and x-halo cells of its cross
constexpr int HALO = YH + XH;
constexpr int OB = NT / 128;             // 1 KB DMA blocks of the own cells of a plane
static_assert(NW == 8 && OB == 4 && TILE <= 128 * NW, "the wave shares below are for 8 waves");
constexpr int LHY = 5 * NT, LHX = LHY + 3 * YH, LEAD = LHX + 3 * XH;  // staged leading plane
constexpr int LU = BY * PX, LV = R * TX; // u rows and v columns of a plane
static_assert(LEAD >= 4 * LU + LV && 5 * TILE >= 6 * LV && TILE >= LU && LV >= LU, "places of the window fill");
enum { RRHO = 0, RMX, RMY, RMZ, RE, RNF };
enum { VU = 0, VV, VW, VT, VP, VNF };

// Taps are read one by one: the compiler otherwise pairs them into ds_read2_b64, which moves
// 128 bytes per cycle where ds_read_b64 moves 240 (measured, eight waves).
template <typename T>
using lds_tap = const volatile __attribute__((address_space(3))) T;

__device__ __forceinline__ void dma16(const double *src, unsigned off, lds_double *lds)
{
    __builtin_amdgcn_global_load_lds((const void *)((const char *)src + off), (lds_void *)lds, 16, 0, 0);
}

// A lane's element of a plane: uniform plane pointer, 32-bit byte offset (a plane is below
// 4 GiB), so that the access is one scalar-base instruction.
#define GAS __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ T GAS &at(T *p, unsigned off)
{
    asm volatile("" : "+s"(p));  // kept scalar: folded with the offset it would take a register pair per array
    return *(T GAS *)((const char GAS *)p + off);
}

// Keeps the scheduler from hoisting the LDS reads of later groups above earlier ones, which
// bounds the live registers.
#define FENCE() __builtin_amdgcn_sched_barrier(0)
// Has the values computed where it stands: the compiler would otherwise move arithmetic that
// is used later past the barriers, and keep its operands live instead.
template <typename... T>
__device__ __forceinline__ void pin(T &...v)
{
    (..., [](auto &x) { asm volatile("" : "+v"(x)); }(v));
}
// A thread index that the compiler cannot see through: what is formed from it is formed
// anew where it stands.  Held across the plane loop, the lane's places and offsets would
// push window entries into scratch.
__device__ __forceinline__ unsigned opaque_tid()
{
    unsigned t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t & (NT - 1);
}
// Products of indices and pitches, all below 2^24 (a full 32-bit product takes four times
// the time of a 24-bit one).
__device__ __forceinline__ unsigned mul24(unsigned a, unsigned b) { return __umul24(a, b); }

// The taps of a lane around cell i of an array in LDS.  The lane's byte offset is formed once,
// with the array's place in LDS in it, so that every tap is a constant of at most 64 KB away,
// which an LDS instruction holds; left to itself the compiler forms an address per tap.
// (The index is hidden and not the pointer: a pointer of unknown origin might read what the
// DMA in flight writes, and would wait for it.)  at: where the array lies, a matter of speed
// alone.
template <int at, typename T = double>
struct Taps {
    const __attribute__((address_space(3))) char *a;
    unsigned off;
    __device__ __forceinline__ Taps(const T *array, unsigned i)
        : a((const __attribute__((address_space(3))) char *)array), off(i * (unsigned)sizeof(T) + at)
    {
        asm volatile("" : "+v"(off));
    }
    __device__ __forceinline__ T operator[](int i) const
    {
        return *(lds_tap<T> *)(a + (off + (unsigned)((int)sizeof(T) * i - at)));
    }
};

// One tap pair (+m, -m) of a sum of differences, in the reference's order: the sum of a term
// begins with its first tap pair.
template <bool FIRST, typename T>
__device__ __forceinline__ void tap(T &s, T t)
{
    s = FIRST ? t : s + t;
}

// hypterm's tap pair in one direction: n the momentum along it, a and b the others, v the
// velocity along it, p the pressure of the momentum flux and q that of the energy flux (where
// the one is taken relative to a reference); sums s of rho, n, a, b, E (cpu/hypterm.cpp:43-90).
template <bool FIRST, typename T>
__device__ __forceinline__ void hyp_tap(T c, T n1, T n0, T a1, T a0, T b1, T b0, T e1, T e0, T p1, T p0, T q1, T q0,
                                        T v1, T v0, T (&s)[5])
{
    tap<FIRST>(s[0], c * (n1 - n0));
    tap<FIRST>(s[1], c * (n1 * v1 - n0 * v0 + (p1 - p0)));
    tap<FIRST>(s[2], c * (a1 * v1 - a0 * v0));
    tap<FIRST>(s[3], c * (b1 * v1 - b0 * v0));
    tap<FIRST>(s[4], c * (e1 * v1 - e0 * v0 + (q1 * v1 - q0 * v0)));
}

}  // namespace

}  // namespace cns
