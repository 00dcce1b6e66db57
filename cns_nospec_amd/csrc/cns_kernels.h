// cns_kernels.h -- host launchers of the CNS_NoSpec HIP kernels (internal).
#pragma once

#include "cns_common.h"

namespace cns {

// A set of n boxes of one geometry stored back to back: box b of an array starts
// b * stride doubles after box 0, with stride su for 5-component ghosted arrays (U),
// sq for 6-component ghosted ones (Q), sc for 5-component interior ones (D, F).  The
// default is a single box.
struct BoxSet {
    int n = 1;
    int64_t su = 0, sq = 0, sc = 0;
};
constexpr int kOneBox[3] = {1, 1, 1};
inline BoxSet box_set(const Geom &g, int n)
{
    BoxSet b;
    b.n = n;
    b.su = NC * g.cg;
    b.sq = NQ * g.cg;
    b.sc = NC * g.c;
    return b;
}

// Ghost shell of u (5 components) and, when not null, of q (6), closed-form periodic image
// (cns_kernels.hip).
hipError_t launch_fill_boundary(const Geom &g, double *u, double *q, hipStream_t s);
// The periodic fill of a domain of nb[0] x nb[1] x nb[2] boxes (box b = I + nb[0]*(J +
// nb[1]*K) at cell origin (I*n0, J*n1, K*n2)): each ghost cell of each box gets the
// domain cell at the periodic image of its global index, from whichever box holds
// it (multifab_fill_boundary, fortran90/advance.f90:81).  With one box it equals
// launch_fill_boundary.
hipError_t launch_domain_fill(const Geom &g, const BoxSet &bs, const int nb[3], double *u, double *q, hipStream_t s);

// Resets a Courant accumulator slot to the bits of max(init, 0) (cns_kernels.hip).
hipError_t launch_courno_reset(unsigned long long *acc, double init, hipStream_t s);

// ctoprim over the ghosted box; acc != nullptr adds the Courant max reduction.
hipError_t launch_ctoprim(const Geom &g, const double *u, double *q, unsigned long long *acc,
                          double dx0, double dx1, double dx2, hipStream_t s);

// The device words and the pinned host words of a StepDt.  step_dt_begin() before each step clears
// acc while it is fresh, that is until a step has run outside a capture (a captured first step
// takes the clearing launch with it: its graph may never run).
hipError_t step_dt_begin(unsigned long long *acc, bool &fresh, hipStream_t s);
hipError_t step_dt_alloc(unsigned long long **acc, double **dt, double **courno, double **host);
void step_dt_free(unsigned long long *acc, double *host);
// sd.dt = cfl / max(acc, 1e-50) and the Courant number; acc back to zero.
hipError_t launch_courno_to_dt(const StepDt &sd, hipStream_t s);

// RK3 stage update; dt from dt_dev when non-null, else dt_host.
hipError_t launch_rk_update(const Geom &g, int phase, double *u, double *unew, const double *d,
                            const double *f, const double *dt_dev, double dt_host, hipStream_t s);

// Reference-order restatements, one thread per output cell, direct global loads
// (cns_kernels.hip).  Used by the free-standing ABI entry points' cross-check path.
hipError_t launch_hypterm_direct(const Geom &g, const double *cons, const double *q, double *flux,
                                 double dxi0, double dxi1, double dxi2, hipStream_t s);
hipError_t launch_diffterm_direct(const Geom &g, const double *q, double *difflux, double dxi0,
                                  double dxi1, double dxi2, double eta, double alam, hipStream_t s);

// z-marching, LDS-tiled stencil kernels (cns_stencil.hip).
hipError_t launch_hypterm_tiled(const Geom &g, const double *cons, const double *q, double *flux,
                                double dxi0, double dxi1, double dxi2, hipStream_t s);
// hypterm with the RK3 stage update of its cell fused in: flux as cns_hypterm, then
// phase 1: out = cons + dt(d+f); 2: out = 3/4 base + 1/4(cons + dt(d+f));
// 3: out = 1/3 base + 2/3(cons + dt(d+f)).  out must not alias cons.
hipError_t launch_hypterm_rk(const Geom &g, const double *cons, const double *q, double *flux,
                             double dxi0, double dxi1, double dxi2, const double *d,
                             const double *base, double *out, const double *dt_dev, int phase,
                             hipStream_t s);
hipError_t launch_diffterm_tiled(const Geom &g, const double *q, double *difflux, double dxi0,
                                 double dxi1, double dxi2, double eta, double alam, hipStream_t s);

// DMA-pipelined z-marching stencils (cns_stencil_pipe.hip).  Every array must be
// 16-byte aligned (pipe_aligned).  diffterm reads wz, a one-component ghosted array filled by
// launch_wz from the same q.
bool pipe_aligned(const void *p);
hipError_t launch_hypterm_pipe(const Geom &g, const double *cons, const double *q, double *flux, const double dxi[3],
                               hipStream_t s);
// The same with stage 1's update in place of storing the flux: out = cons + dt (d + flux).
hipError_t launch_hypterm_pipe_rk1(const Geom &g, const double *cons, const double *q, const double dxi[3],
                                   const double *d, double *out, const double *dt_dev, hipStream_t s);
hipError_t launch_wz(const Geom &g, const double *q, double *wz, double dxi2, hipStream_t s);
hipError_t launch_diffterm_pipe(const Geom &g, const double *q, const double *wz, double *difflux,
                                double dxi0, double dxi1, double dxi2, double eta, double alam,
                                hipStream_t s);

// The start of a fused step in one launch: the periodic ghosts of u (every box of the set) and
// the Courant maximum of its interior into acc.  The two touch different cells.
hipError_t launch_fill_courno(const Geom &g, double *u, unsigned long long *acc, double dx0, double dx1,
                              double dx2, hipStream_t s, const BoxSet &bs = BoxSet(), const int nb[3] = kOneBox);
// One RK stage in one kernel (cns_stage.hip): out = the SSP-RK3 update of phase 1..3 of the
// ghosted state cons with base U^n (phases 2 and 3), its primitives into q (phase 2), D and
// F stored by phase 3.  Every array must be 16-byte aligned; out must not alias cons; the
// geometry must satisfy stage_fits (planes below 4 GiB, pitches below 2^24).
// wrapped (one box; the same array as cons in phases 2 and 3, any in phase 1): the periodic
// box needs no fill between its stages.  Phases 1 and 2 store the x ghosts of out beside its
// interior, phases 2 and 3 read cons at wrapped rows and planes, and phase 3 fills the ghosts
// of cons (which is not const then) and q.  Null: cons has its ghosts filled.
bool stage_fits(const Geom &g);
bool stage_pays(const Geom &g);   // whether a step of separate kernels would be slower
bool stage_wraps(const Geom &g);  // whether a periodic box is stepped without fills between its stages
hipError_t launch_stage(const Geom &g, const double *cons, const double *base, double *out, double *q, double *d,
                        double *f, const StepDt &sd, const double dxi[3], double eta, double alam, int phase,
                        hipStream_t s, const BoxSet &bs = BoxSet(), double *wrapped = nullptr);

}  // namespace cns
