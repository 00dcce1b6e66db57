// cns_fill.h -- the periodic ghost fill of one cell (internal).
#pragma once

#include "cns_common.h"
#include "cns_kernels.h"

namespace cns {

namespace {

// The reference fills the ghost shell in three ordered copy passes (z planes over
// interior i,j; y planes over interior i and all k; x columns over all j,k:
// cpu/helper_functions.cpp:226-262, gpu/util.cu:53-127).  For extents >= NG their
// composition maps every ghost cell to the interior cell at the periodic image
// of all three of its indices, so one pass over the shell copies exactly the same
// values.  The shell is enumerated compactly: first the full rows whose j or k is
// a ghost index (g0 cells each), then the 2*NG ghost cells of each interior row.
//
// One thread per ghost cell, its components' loads all in flight before the first store.
// What bounds it: at small boxes latency, so the index arithmetic is 32-bit with
// precomputed quotients; at large ones the x ghosts, whose four-cell pieces touch
// two 128-byte lines per row and component.
//
// N counts the cells: 32 bits, or 64 with ordinary division for the long thin boxes of the
// free-standing fill that have 2^32 ghost cells or more.
template <typename N>
struct ShellOf {
    FastDiv g0, g1, n1, nbx, nby;
    N plane_rows, elems_a, total;  // rows of the ghost planes; cells of the full rows; all cells
};
using Shell = ShellOf<unsigned>;

template <typename N = unsigned>
inline ShellOf<N> make_shell(const Geom &g, const int nb[3])
{
    ShellOf<N> h;
    h.g0 = fast_div(g.g0);
    h.g1 = fast_div(g.g1);
    h.n1 = fast_div(g.n1);
    h.nbx = fast_div(nb[0]);
    h.nby = fast_div(nb[1]);
    h.plane_rows = (N)(2 * NG) * g.g1;
    h.elems_a = (h.plane_rows + (N)(2 * NG) * g.n2) * g.g0;
    h.total = h.elems_a + (N)(2 * NG) * g.n1 * g.n2;
    return h;
}

__host__ __device__ __forceinline__ unsigned quotient(unsigned n, const FastDiv &by) { return by.div(n); }
__host__ __device__ __forceinline__ uint64_t quotient(uint64_t n, const FastDiv &by) { return n / by.d; }

inline int64_t shell_cells(const Geom &g)
{
    return ((int64_t)2 * NG * g.g1 + (int64_t)2 * NG * g.n2) * g.g0 + (int64_t)2 * NG * g.n1 * g.n2;
}

// Ghost cell e of the enumeration, as (i, j, k).
template <typename N>
__host__ __device__ __forceinline__ void shell_cell(const Geom &g, const ShellOf<N> &h, N e, int &i, int &j, int &k)
{
    if (e < h.elems_a) {
        N r = quotient(e, h.g0);
        i = (int)(e - r * g.g0);
        if (r < h.plane_rows) {
            const int kk = (int)quotient(r, h.g1);
            j = (int)r - kk * g.g1;
            k = kk < NG ? kk : g.n2 + kk;
        } else {
            r -= h.plane_rows;
            const int jj = (int)(r & (2 * NG - 1));
            k = NG + (int)(r / (2 * NG));
            j = jj < NG ? jj : g.n1 + jj;
        }
    } else {
        const N e2 = e - h.elems_a, row = e2 / (2 * NG), kk = quotient(row, h.n1);
        const int ii = (int)(e2 & (2 * NG - 1));
        i = ii < NG ? ii : g.n0 + ii;
        k = NG + (int)kk;
        j = NG + (int)(row - kk * g.n1);
    }
}

// One axis of a ghost cell at index a of box I of nb boxes of n cells: the box (relative
// step dI) and the index there of the cell it is the periodic image of.  Extents are at
// least NG, so that is the neighbouring box.
__device__ __forceinline__ int image(int a, int I, int n, int nb, int &dI)
{
    dI = a < NG ? (I == 0 ? nb - 1 : -1) : (a >= n + NG ? (I == nb - 1 ? 1 - nb : 1) : 0);
    return a < NG ? a + n : (a >= n + NG ? a - n : a);
}

// Ghost cell e of box b of a set of nb[0] x nb[1] x nb[2] boxes (one box: its own images).  Q:
// the components of q as well.  u_x: u's x ghosts of the interior rows too.
template <bool Q, typename N>
__device__ __forceinline__ void fill_cell(const Geom &g, const ShellOf<N> &h, const BoxSet &bs, int nbx, int nby, int nbz,
                                          N e, unsigned b, double *u, double *q, bool u_x = true)
{
    const unsigned r = h.nbx.div(b);
    const int K = (int)h.nby.div(r), J = (int)r - K * nby, I = (int)b - (int)r * nbx;
    int i, j, k, dI, dJ, dK;
    shell_cell(g, h, e, i, j, k);
    const int is = image(i, I, g.n0, nbx, dI), js = image(j, J, g.n1, nby, dJ), ks = image(k, K, g.n2, nbz, dK);
    const int64_t bsrc = (int64_t)b + dI + (int64_t)nbx * (dJ + (int64_t)nby * dK);
    const int64_t dst = gidx(g, i, j, k), src = gidx(g, is, js, ks);
    const double *us = u + bsrc * bs.su + src;
    double *ud = u + b * bs.su + dst;
    const bool fill_u = u_x || e < h.elems_a;
    double v[NC], w[NQ];
    if (fill_u) {
#pragma unroll
        for (int l = 0; l < NC; l++) v[l] = us[l * g.cg];
    }
    if (Q) {
        const double *qs = q + bsrc * bs.sq + src;
#pragma unroll
        for (int l = 0; l < NQ; l++) w[l] = qs[l * g.cg];
    }
    if (fill_u) {
#pragma unroll
        for (int l = 0; l < NC; l++) ud[l * g.cg] = v[l];
    }
    if (Q) {
        double *qd = q + b * bs.sq + dst;
#pragma unroll
        for (int l = 0; l < NQ; l++) qd[l * g.cg] = w[l];
    }
}

}  // namespace

}  // namespace cns
