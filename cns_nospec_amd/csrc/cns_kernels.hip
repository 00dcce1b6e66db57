// cns_kernels.hip -- streaming kernels of the CNS_NoSpec step (gfx950):
// periodic ghost fill, ctoprim with the Courant max-reduction, the RK3 stage
// update, and the reference-order direct-load stencils used to cross-check the
// tiled ones.
//
// Every kernel keeps the reference's per-cell operation order; the library is
// compiled with -ffp-contract=off, so results are bit-identical to the
// reference cpu/ path (which g++ -O2 builds without FMA).
#include <algorithm>
#include <bitset>
#include <functional>
#include <mutex>

#include "cns_kernels.h"
#include "cns_fill.h"

namespace cns {

namespace {

constexpr int kStreamBlock = 256;

inline int stream_grid(int64_t work, int per_thread = 4)
{
    int64_t blocks = (work + (int64_t)kStreamBlock * per_thread - 1) / ((int64_t)kStreamBlock * per_thread);
    if (blocks < 1) blocks = 1;
    if (blocks > 65536) blocks = 65536;
    return (int)blocks;
}

// ------------------------------------------------------------------ ghost fill (cns_fill.h)
template <bool Q>
__global__ void __launch_bounds__(kStreamBlock)
fill_kernel(Geom g, Shell h, BoxSet bs, int nbx, int nby, int nbz, double *__restrict__ u, double *__restrict__ q)
{
    const unsigned e = blockIdx.x * kStreamBlock + threadIdx.x;
    if (e < h.total) fill_cell<Q>(g, h, bs, nbx, nby, nbz, e, blockIdx.y, u, q);
}

// 2^32 ghost cells of a box and more
template <bool Q>
__global__ void __launch_bounds__(kStreamBlock)
fill_long_kernel(Geom g, ShellOf<uint64_t> h, BoxSet bs, int nbx, int nby, int nbz, double *__restrict__ u,
                 double *__restrict__ q)
{
    for (uint64_t e = (uint64_t)blockIdx.x * kStreamBlock + threadIdx.x; e < h.total; e += (uint64_t)gridDim.x * kStreamBlock)
        fill_cell<Q>(g, h, bs, nbx, nby, nbz, e, blockIdx.y, u, q);
}

// -------------------------------------------------------------------- courno
__global__ void courno_reset_kernel(unsigned long long *acc, double init)
{
    acc[0] = init > 0.0 ? (unsigned long long)__double_as_longlong(init) : 0ull;
}

__global__ void courno_to_dt_kernel(StepDt sd)
{
    double courno;
    const double dt = courno_dt(sd.acc, sd.cfl, courno);
    step_dt_store(sd, dt, courno);
    sd.acc[0] = 0ull;
}

// ------------------------------------------------------------------- ctoprim
// Per ghosted cell (cpu/ctoprim.cpp:27-44):
//   rhoinv = 1/rho; q = (rho, mx*rhoinv, my*rhoinv, mz*rhoinv, (g-1)*eint*rho, eint/CV),
//   eint = E*rhoinv - 0.5*(u^2+v^2+w^2).
// With COURNO, per interior cell (cpu/ctoprim.cpp:48-63): c = sqrt(g*p/rho),
// cour_d = (c+|u_d|)/dx_d; the block's maximum goes to acc with one atomic.
// The grid strides over the padded linear index space, so one wave touches 64
// consecutive doubles of a row (coalesced); lanes on padding skip.
template <bool COURNO>
__global__ void __launch_bounds__(kStreamBlock)
ctoprim_kernel(Geom g, const double *__restrict__ u, double *__restrict__ q,
               unsigned long long *__restrict__ acc, double dx0, double dx1, double dx2)
{
    const int64_t total = (int64_t)g.g2 * g.pg;
    const int64_t cg = g.cg;
    unsigned long long cmax = 0ull;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t row = e / g.xg;
        const int i = (int)(e - row * g.xg);
        if (i >= g.g0) continue;
        const double rho = u[e];
        double qu, qv, qw, eint, p;
        ctoprim_cell(rho, u[e + cg], u[e + 2 * cg], u[e + 3 * cg], u[e + 4 * cg], qu, qv, qw, eint, p);
        q[e] = rho;
        q[e + cg] = qu;
        q[e + 2 * cg] = qv;
        q[e + 3 * cg] = qw;
        q[e + 4 * cg] = p;
        q[e + 5 * cg] = eint / CV;
        if (COURNO) {
            const int k = (int)(row / g.g1);
            const int j = (int)(row - (int64_t)k * g.g1);
            if (i >= NG && i < g.n0 + NG && j >= NG && j < g.n1 + NG && k >= NG && k < g.n2 + NG) {
                const double c = sqrt(GAMMA * p / rho);
                const double courx = (c + fabs(qu)) / dx0;
                const double coury = (c + fabs(qv)) / dx1;
                const double courz = (c + fabs(qw)) / dx2;
                unsigned long long b = courno_bits(courx);
                unsigned long long by = courno_bits(coury);
                unsigned long long bz = courno_bits(courz);
                b = b > by ? b : by;
                b = b > bz ? b : bz;
                cmax = cmax > b ? cmax : b;
            }
        }
    }
    if (COURNO) {
        __shared__ unsigned long long wmax[kStreamBlock / 64];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            unsigned long long o = __shfl_xor(cmax, off);
            cmax = cmax > o ? cmax : o;
        }
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        if (lane == 0) wmax[wave] = cmax;
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned long long m = wmax[0];
            for (int w = 1; w < kStreamBlock / 64; w++) m = m > wmax[w] ? m : wmax[w];
            atomicMax(acc, m);
        }
    }
}

// ------------------------------------------------------------------ RK update
// cpu/advance.cpp:78-85 (phase 1), :110-119 (phase 2), :144-153 (phase 3).
// HBM-bound at large boxes (256^3 0.67 ms, 4.7 TB/s).  All operands of a cell are loaded before its
// first store: u and unew are read and written at the same places, so the compiler would keep loads
// behind stores and a cell wait five times (64^3 14.0 -> 9.4 us, with one quotient a thread).
template <int PHASE>
__global__ void __launch_bounds__(kStreamBlock)
rk_update_kernel(Geom g, double *__restrict__ u, double *__restrict__ unew, const double *__restrict__ d,
                 const double *__restrict__ f, const double *__restrict__ dt_dev, double dt_host, FastDiv by_x)
{
    const double dt = dt_dev ? dt_dev[0] : dt_host;
    const unsigned in = blockIdx.x * kStreamBlock + threadIdx.x;  // of the plane
    const int j = (int)by_x.div(in), i = (int)(in - (unsigned)j * by_x.d);
    if (j >= g.n1 || i >= g.n0) return;
    for (int k = blockIdx.y; k < g.n2; k += gridDim.y) {
        const int64_t o = gidx(g, i + NG, j + NG, k + NG), e = (int64_t)k * g.p + in;
        double a[NC], b[NC], x[NC], y[NC];
#pragma unroll
        for (int l = 0; l < NC; l++) {
            a[l] = u[l * g.cg + o];
            b[l] = PHASE == 1 ? 0.0 : unew[l * g.cg + o];
            x[l] = d[l * g.c + e];
            y[l] = f[l * g.c + e];
        }
#pragma unroll
        for (int l = 0; l < NC; l++) {
            const int64_t go = l * g.cg + o;
            if (PHASE == 1)
                unew[go] = a[l] + dt * (x[l] + y[l]);
            else if (PHASE == 2)
                unew[go] = ThreeQuarters * a[l] + OneQuarter * (b[l] + dt * (x[l] + y[l]));
            else
                u[go] = OneThird * a[l] + TwoThirds * (b[l] + dt * (x[l] + y[l]));
        }
    }
}

// ---------------------------------------------------------------- Courant number
// The Courant maximum of a state's interior cells (cpu/ctoprim.cpp:42-69), without storing
// its primitives, into acc (one 64-bit atomicMax per block).  A thread takes every
// (grid size)-th cell of the interior, so a wave reads 64 consecutive cells of a row but for
// the row ends: HBM-bound at large boxes (512^3 1.0 ms, 5.4 TB/s).
// The first `cb` blocks of a box do this; the others fill u's ghosts, one cell a thread: the two
// touch different cells, and a step of a small box is a few launches long.
__global__ void __launch_bounds__(kStreamBlock)
fill_courno_kernel(Geom g, double *__restrict__ u, unsigned long long *__restrict__ acc, double dx0, double dx1,
                   double dx2, FastDiv by_n0, FastDiv by_n1, unsigned cells, unsigned cb, Shell h, BoxSet bs, int nbx,
                   int nby, int nbz)
{
    if (blockIdx.x >= cb) {
        const unsigned e = (blockIdx.x - cb) * kStreamBlock + threadIdx.x;
        if (e < h.total) fill_cell<false>(g, h, bs, nbx, nby, nbz, e, blockIdx.y, u, nullptr);
        return;
    }
    u += blockIdx.y * bs.su;  // box of a box set
    const int64_t cg = g.cg;
    unsigned long long cmax = 0ull;
    for (unsigned n = blockIdx.x * kStreamBlock + threadIdx.x; n < cells; n += cb * kStreamBlock) {
        const unsigned r = by_n0.div(n), k = by_n1.div(r);
        const int64_t e = gidx(g, (int)(n - r * g.n0) + NG, (int)(r - k * g.n1) + NG, (int)k + NG);
        const double rho = u[e];
        double qu, qv, qw, eint, p;
        ctoprim_cell(rho, u[e + cg], u[e + 2 * cg], u[e + 3 * cg], u[e + 4 * cg], qu, qv, qw, eint, p);
        const double c = sqrt(GAMMA * p / rho);
        unsigned long long b = courno_bits((c + fabs(qu)) / dx0);
        const unsigned long long by = courno_bits((c + fabs(qv)) / dx1);
        const unsigned long long bz = courno_bits((c + fabs(qw)) / dx2);
        b = b > by ? b : by;
        b = b > bz ? b : bz;
        cmax = cmax > b ? cmax : b;
    }
    __shared__ unsigned long long wmax[kStreamBlock / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long o = __shfl_xor(cmax, off);
        cmax = cmax > o ? cmax : o;
    }
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = cmax;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long m = wmax[0];
        for (int w = 1; w < kStreamBlock / 64; w++) m = m > wmax[w] ? m : wmax[w];
        atomicMax(acc, m);
    }
}

// ------------------------------------------------- direct-load stencils
__device__ __forceinline__ double d1(const double *__restrict__ f, int64_t o, int64_t s)
{
    return ALP * (f[o + s] - f[o - s]) + BET * (f[o + 2 * s] - f[o - 2 * s])
           + GAM * (f[o + 3 * s] - f[o - 3 * s]) + DEL * (f[o + 4 * s] - f[o - 4 * s]);
}

__device__ __forceinline__ double d2(const double *__restrict__ f, int64_t o, int64_t s)
{
    return CENTER * f[o] + OFF1 * (f[o + s] + f[o - s]) + OFF2 * (f[o + 2 * s] + f[o - 2 * s])
           + OFF3 * (f[o + 3 * s] + f[o - 3 * s]) + OFF4 * (f[o + 4 * s] + f[o - 4 * s]);
}

// Sums of one direction of cpu/hypterm.cpp (x :33-90, y :101-147, z :158-204) before *dxinv.
template <int DIR>
__device__ __forceinline__ void hyp_sums(const double *__restrict__ cons,
                                         const double *__restrict__ q, int64_t o, int64_t s,
                                         int64_t cg, double A[5])
{
    constexpr int qn = QU + DIR, mn = IMX + DIR;
    const double *cm = cons + mn * cg;
    const double *un = q + qn * cg;
    const double *pr = q + QPRES * cg;
#define UN(m) un[o + (m) * s]
#define P(m) pr[o + (m) * s]
#define CC(l, m) cons[(l) * cg + o + (m) * s]
    A[IRHO] = ALP * (cm[o + s] - cm[o - s]) + BET * (cm[o + 2 * s] - cm[o - 2 * s])
              + GAM * (cm[o + 3 * s] - cm[o - 3 * s]) + DEL * (cm[o + 4 * s] - cm[o - 4 * s]);
#pragma unroll
    for (int l = IMX; l <= IMZ; l++) {
        if (l == mn)
            A[l] = ALP * (CC(l, 1) * UN(1) - CC(l, -1) * UN(-1) + (P(1) - P(-1)))
                   + BET * (CC(l, 2) * UN(2) - CC(l, -2) * UN(-2) + (P(2) - P(-2)))
                   + GAM * (CC(l, 3) * UN(3) - CC(l, -3) * UN(-3) + (P(3) - P(-3)))
                   + DEL * (CC(l, 4) * UN(4) - CC(l, -4) * UN(-4) + (P(4) - P(-4)));
        else
            A[l] = ALP * (CC(l, 1) * UN(1) - CC(l, -1) * UN(-1))
                   + BET * (CC(l, 2) * UN(2) - CC(l, -2) * UN(-2))
                   + GAM * (CC(l, 3) * UN(3) - CC(l, -3) * UN(-3))
                   + DEL * (CC(l, 4) * UN(4) - CC(l, -4) * UN(-4));
    }
    A[IENE] = ALP * (CC(IENE, 1) * UN(1) - CC(IENE, -1) * UN(-1) + (P(1) * UN(1) - P(-1) * UN(-1)))
              + BET * (CC(IENE, 2) * UN(2) - CC(IENE, -2) * UN(-2) + (P(2) * UN(2) - P(-2) * UN(-2)))
              + GAM * (CC(IENE, 3) * UN(3) - CC(IENE, -3) * UN(-3) + (P(3) * UN(3) - P(-3) * UN(-3)))
              + DEL * (CC(IENE, 4) * UN(4) - CC(IENE, -4) * UN(-4) + (P(4) * UN(4) - P(-4) * UN(-4)));
#undef UN
#undef P
#undef CC
}

// cpu/hypterm.cpp:11-209, one thread per interior cell, x then y then z.
__global__ void __launch_bounds__(256)
hypterm_direct_kernel(Geom g, const double *__restrict__ cons, const double *__restrict__ q,
                      double *__restrict__ flux, double dxi0, double dxi1, double dxi2)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= g.n0 || j >= g.n1) return;
    const int64_t o = gidx(g, i + NG, j + NG, k + NG);
    const int64_t fo = iidx(g, i, j, k);
    double A[5], F[5];
    hyp_sums<0>(cons, q, o, 1, g.cg, A);
#pragma unroll
    for (int l = 0; l < NC; l++) F[l] = -(A[l]) * dxi0;
    hyp_sums<1>(cons, q, o, g.xg, g.cg, A);
#pragma unroll
    for (int l = 0; l < NC; l++) F[l] = F[l] - (A[l]) * dxi1;
    hyp_sums<2>(cons, q, o, g.pg, g.cg, A);
#pragma unroll
    for (int l = 0; l < NC; l++) F[l] = F[l] - (A[l]) * dxi2;
#pragma unroll
    for (int l = 0; l < NC; l++) flux[l * g.c + fo] = F[l];
}

// cpu/diffterm.cpp:22-320, one thread per interior cell.  The first derivatives
// the reference stores in nine temporaries are recomputed at each use with the
// same expression, so each value is the same double.
__global__ void __launch_bounds__(256)
diffterm_direct_kernel(Geom g, const double *__restrict__ q, double *__restrict__ difflux,
                       double dxi0, double dxi1, double dxi2, double eta, double alam)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= g.n0 || j >= g.n1) return;
    const int64_t o = gidx(g, i + NG, j + NG, k + NG);
    const int64_t fo = iidx(g, i, j, k);
    const int64_t sx = 1, sy = g.xg, sz = g.pg, c = g.c;
    const double *qU = q + QU * g.cg, *qV = q + QV * g.cg, *qW = q + QW * g.cg;
    const double *qT = q + QTEMP * g.cg;

#define UX(p) (d1(qU, (p), sx) * dxi0)
#define VY(p) (d1(qV, (p), sy) * dxi1)
#define WZ(p) (d1(qW, (p), sz) * dxi2)
#define D1OF(F, s, dxi) \
    ((ALP * (F(o + (s)) - F(o - (s))) + BET * (F(o + 2 * (s)) - F(o - 2 * (s))) \
      + GAM * (F(o + 3 * (s)) - F(o - 3 * (s))) + DEL * (F(o + 4 * (s)) - F(o - 4 * (s)))) * (dxi))

    const double uxx = d2(qU, o, sx) * (dxi0 * dxi0);
    const double uyy = d2(qU, o, sy) * (dxi1 * dxi1);
    const double uzz = d2(qU, o, sz) * (dxi2 * dxi2);
    const double vyx = D1OF(VY, sx, dxi0);
    const double wzx = D1OF(WZ, sx, dxi0);
    const double dmx = eta * (FourThirds * uxx + uyy + uzz + OneThird * (vyx + wzx));

    const double vxx = d2(qV, o, sx) * (dxi0 * dxi0);
    const double vyy = d2(qV, o, sy) * (dxi1 * dxi1);
    const double vzz = d2(qV, o, sz) * (dxi2 * dxi2);
    const double uxy = D1OF(UX, sy, dxi1);
    const double wzy = D1OF(WZ, sy, dxi1);
    const double dmy = eta * (vxx + FourThirds * vyy + vzz + OneThird * (uxy + wzy));

    const double wxx = d2(qW, o, sx) * (dxi0 * dxi0);
    const double wyy = d2(qW, o, sy) * (dxi1 * dxi1);
    const double wzz = d2(qW, o, sz) * (dxi2 * dxi2);
    const double uxz = D1OF(UX, sz, dxi2);
    const double vyz = D1OF(VY, sz, dxi2);
    const double dmz = eta * (wxx + wyy + FourThirds * wzz + OneThird * (uxz + vyz));

    const double txx = d2(qT, o, sx) * (dxi0 * dxi0);
    const double tyy = d2(qT, o, sy) * (dxi1 * dxi1);
    const double tzz = d2(qT, o, sz) * (dxi2 * dxi2);
    const double ux = UX(o), vy = VY(o), wz = WZ(o);
    const double uy = d1(qU, o, sy) * dxi1, uz = d1(qU, o, sz) * dxi2;
    const double vx = d1(qV, o, sx) * dxi0, vz = d1(qV, o, sz) * dxi2;
    const double wx = d1(qW, o, sx) * dxi0, wy = d1(qW, o, sy) * dxi1;
    const double divu = TwoThirds * (ux + vy + wz);
    const double tauxx = 2.E0 * ux - divu;
    const double tauyy = 2.E0 * vy - divu;
    const double tauzz = 2.E0 * wz - divu;
    const double tauxy = uy + vx;
    const double tauxz = uz + wx;
    const double tauyz = vz + wy;
    double mechwork = tauxx * ux + tauyy * vy + tauzz * wz + (tauxy * tauxy) + (tauxz * tauxz)
                      + (tauyz * tauyz);
    mechwork = eta * mechwork + dmx * qU[o] + dmy * qV[o] + dmz * qW[o];

    difflux[fo] = 0.0E0;
    difflux[fo + IMX * c] = dmx;
    difflux[fo + IMY * c] = dmy;
    difflux[fo + IMZ * c] = dmz;
    difflux[fo + IENE * c] = alam * (txx + tyy + tzz) + mechwork;
#undef UX
#undef VY
#undef WZ
#undef D1OF
}

}  // namespace

// ------------------------------------------------------------------ launchers
hipError_t launch_domain_fill(const Geom &g, const BoxSet &bs, const int nb[3], double *u, double *q, hipStream_t s)
{
    const int64_t total = shell_cells(g);
    if (bs.n != nb[0] * nb[1] * nb[2] || bs.n < 1 || bs.n > 65535) return hipErrorInvalidValue;
    if (total > 0xffffffffll - kStreamBlock) {
        const ShellOf<uint64_t> h = make_shell<uint64_t>(g, nb);
        const dim3 grid(1u << 16, (unsigned)bs.n);
        if (q)
            fill_long_kernel<true><<<grid, kStreamBlock, 0, s>>>(g, h, bs, nb[0], nb[1], nb[2], u, q);
        else
            fill_long_kernel<false><<<grid, kStreamBlock, 0, s>>>(g, h, bs, nb[0], nb[1], nb[2], u, nullptr);
        return hipGetLastError();
    }
    const Shell h = make_shell(g, nb);
    const dim3 grid((unsigned)((total + kStreamBlock - 1) / kStreamBlock), (unsigned)bs.n);
    if (q)
        fill_kernel<true><<<grid, kStreamBlock, 0, s>>>(g, h, bs, nb[0], nb[1], nb[2], u, q);
    else
        fill_kernel<false><<<grid, kStreamBlock, 0, s>>>(g, h, bs, nb[0], nb[1], nb[2], u, nullptr);
    return hipGetLastError();
}

hipError_t launch_fill_boundary(const Geom &g, double *u, double *q, hipStream_t s)
{
    return launch_domain_fill(g, BoxSet(), kOneBox, u, q, s);
}

hipError_t launch_courno_reset(unsigned long long *acc, double init, hipStream_t s)
{
    courno_reset_kernel<<<1, 1, 0, s>>>(acc, init);
    return hipGetLastError();
}

hipError_t launch_fill_courno(const Geom &g, double *u, unsigned long long *acc, double dx0, double dx1,
                              double dx2, hipStream_t s, const BoxSet &bs, const int nb[3])
{
    if (bs.n != nb[0] * nb[1] * nb[2] || bs.n < 1 || bs.n > 65535) return hipErrorInvalidValue;
    // Each block ends in an atomic on one address, about 20 ns apiece one after the other, so
    // small boxes take 256 blocks (128^3: 57 us with 4096 blocks, 26 with 512) and large ones up
    // to 1024, which their bandwidth needs (512^3: 1.76 / 1.13 / 1.00 / 1.02 ms with 256 / 512 /
    // 1024 / 2048): 16 cells a thread or more in between.
    const int64_t cells = (int64_t)g.n0 * g.n1 * g.n2, all = cells * bs.n;
    const int64_t total = shell_cells(g);
    if (cells > 0xffffffffll - 1024ll * kStreamBlock || total > 0xffffffffll - kStreamBlock) return hipErrorInvalidValue;
    int64_t most = all / (16 * kStreamBlock);
    most = (most < 256 ? 256 : (most > 1024 ? 1024 : most)) / bs.n;
    int64_t gx = (cells + kStreamBlock - 1) / kStreamBlock;
    if (gx > most) gx = most;
    if (gx < 1) gx = 1;
    const unsigned fb = (unsigned)((total + kStreamBlock - 1) / kStreamBlock);
    fill_courno_kernel<<<dim3((unsigned)gx + fb, (unsigned)bs.n), kStreamBlock, 0, s>>>(
        g, u, acc, dx0, dx1, dx2, fast_div(g.n0), fast_div(g.n1), (unsigned)cells, (unsigned)gx, make_shell(g, nb), bs,
        nb[0], nb[1], nb[2]);
    return hipGetLastError();
}

hipError_t launch_ctoprim(const Geom &g, const double *u, double *q, unsigned long long *acc,
                          double dx0, double dx1, double dx2, hipStream_t s)
{
    const int64_t total = (int64_t)g.g2 * g.pg;
    const int grid = stream_grid(total, 8);
    if (acc)
        ctoprim_kernel<true><<<grid, kStreamBlock, 0, s>>>(g, u, q, acc, dx0, dx1, dx2);
    else
        ctoprim_kernel<false><<<grid, kStreamBlock, 0, s>>>(g, u, q, nullptr, dx0, dx1, dx2);
    return hipGetLastError();
}

hipError_t launch_courno_to_dt(const StepDt &sd, hipStream_t s)
{
    courno_to_dt_kernel<<<1, 1, 0, s>>>(sd);
    return hipGetLastError();
}

// Pinned words for dt and courno of a context: one page for the process, in slots that are given
// back, since pinning memory takes longer than all else of a context's creation.  More contexts
// than slots pin their own.
namespace {
struct HostWords {
    static constexpr int kSlots = 256;
    std::mutex mu;
    double *page = nullptr;
    std::bitset<kSlots> used;
};
HostWords g_words;

hipError_t host_words(double **out)
{
    std::lock_guard<std::mutex> lock(g_words.mu);
    if (!g_words.page) {
        const hipError_t e = hipHostMalloc((void **)&g_words.page, HostWords::kSlots * 2 * sizeof(double), hipHostMallocPortable);
        if (e) {
            g_words.page = nullptr;
            return e;
        }
    }
    for (int i = 0; i < HostWords::kSlots; i++)
        if (!g_words.used[i]) {
            g_words.used[i] = true;
            *out = g_words.page + 2 * i;
            return hipSuccess;
        }
    return hipHostMalloc((void **)out, 2 * sizeof(double), hipHostMallocPortable);
}

void host_words_free(double *p)
{
    std::lock_guard<std::mutex> lock(g_words.mu);
    const std::less<const double *> before;
    if (g_words.page && !before(p, g_words.page) && before(p, g_words.page + 2 * HostWords::kSlots))
        g_words.used[(p - g_words.page) / 2] = false;
    else
        (void)hipHostFree(p);
}
}  // namespace

hipError_t step_dt_alloc(unsigned long long **acc, double **dt, double **courno, double **host)
{
    *host = nullptr;
    unsigned long long *blk = nullptr;
    hipError_t e = hipMalloc((void **)&blk, 4 * sizeof(double));
    if (!e) e = host_words(host);
    if (e) {
        (void)hipGetLastError();
        step_dt_free(blk, *host);
        return e;
    }
    *acc = blk;
    *dt = (double *)blk + 1;
    *courno = (double *)blk + 2;
    return hipSuccess;
}

hipError_t step_dt_begin(unsigned long long *acc, bool &fresh, hipStream_t s)
{
    if (!fresh) return hipSuccess;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(s, &st);
    if (!e) e = launch_courno_reset(acc, 0.0, s);
    if (!e && st == hipStreamCaptureStatusNone) fresh = false;
    return e;
}

// (The device is idle once hipFree returns: nothing writes to the host words any more.)
void step_dt_free(unsigned long long *acc, double *host)
{
    if (acc) (void)hipFree(acc);
    if (host) host_words_free(host);
}

hipError_t launch_rk_update(const Geom &g, int phase, double *u, double *unew, const double *d,
                            const double *f, const double *dt_dev, double dt_host, hipStream_t s)
{
    if (g.p > 0x7fffffff) return hipErrorInvalidValue;
    // A thread takes one place of the plane in every (grid y)-th plane, so that its row and column
    // cost one quotient by a launch constant in all.
    const int64_t gx = (g.p + kStreamBlock - 1) / kStreamBlock, each = std::max<int64_t>(1, gx * g.n2 / 16384);
    const dim3 grid((unsigned)gx, (unsigned)std::min<int64_t>(65535, (g.n2 + each - 1) / each));
    const FastDiv by_x = fast_div((unsigned)g.x);
    switch (phase) {
    case 1: rk_update_kernel<1><<<grid, kStreamBlock, 0, s>>>(g, u, unew, d, f, dt_dev, dt_host, by_x); break;
    case 2: rk_update_kernel<2><<<grid, kStreamBlock, 0, s>>>(g, u, unew, d, f, dt_dev, dt_host, by_x); break;
    case 3: rk_update_kernel<3><<<grid, kStreamBlock, 0, s>>>(g, u, unew, d, f, dt_dev, dt_host, by_x); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_hypterm_direct(const Geom &g, const double *cons, const double *q, double *flux,
                                 double dxi0, double dxi1, double dxi2, hipStream_t s)
{
    dim3 block(64, 4, 1), grid((g.n0 + 63) / 64, (g.n1 + 3) / 4, g.n2);
    hypterm_direct_kernel<<<grid, block, 0, s>>>(g, cons, q, flux, dxi0, dxi1, dxi2);
    return hipGetLastError();
}

hipError_t launch_diffterm_direct(const Geom &g, const double *q, double *difflux, double dxi0,
                                  double dxi1, double dxi2, double eta, double alam, hipStream_t s)
{
    dim3 block(64, 4, 1), grid((g.n0 + 63) / 64, (g.n1 + 3) / 4, g.n2);
    diffterm_direct_kernel<<<grid, block, 0, s>>>(g, q, difflux, dxi0, dxi1, dxi2, eta, alam);
    return hipGetLastError();
}

}  // namespace cns
