"""Workloads of the CNS time step that its speed is judged on, each through the public
entry points a program calls: the plain step (eager and captured in a graph), the
reference's CGS deck, the per-kernel operators composed as the reference's main loop, a
multi-box domain, the batched engine in both precisions, and a server's admit / step /
retire cycle.

``listed`` names them, ``draw`` gives more of the same ranges, ``prepare`` makes what the
program holds before the call, ``run`` is one pass, ``work`` the bytes and operations
the pass cannot do without, and ``exact`` the same outputs from plain torch in float64 (no
code of this package): periodic arrays without ghosts, differenced with ``torch.roll``.
"""
import math

import numpy as np
import torch

from cns_nospec_amd import batch, domain, ops
from cns_nospec_amd.layout import NC, NQ, BoxLayout

NG = 4
ETA, ALAM = 1.8e-4, 1.5e2  # the reference's defaults
SIDE = 0.2                 # edge of the periodic domain
GAMMA, CV = 1.4, 8.3333333333e6
# 8th-order central differences
FIRST = (0.8, -0.2, 4.0 / 105.0, -1.0 / 280.0)
SECOND = (-205.0 / 72.0, 8.0 / 5.0, -0.2, 8.0 / 315.0, -1.0 / 560.0)
# flops of one cell in one RK stage: primitives, hypterm, diffterm, update
STAGE_FLOPS = 16 + 363 + 393 + 20


def cfl_of(nmax):
    """cfl 0.5 is the reference's default; with its viscosity the explicit step is unstable
    above about 300 cells a side, so finer boxes are run at half of it."""
    return 0.5 if nmax <= 256 else 0.25


def step_case(name, n, steps=1, mach=0.085, kind="step"):
    return {"name": name, "kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "steps": steps, "mach": mach}


def listed():
    return [
        # the smallest call: one step of a 16^3 box, dt to the host (the reference's 16^3 test
        # problem); launches and the wait for dt are all there is
        step_case("step 16^3", (16, 16, 16)),
        # a small box driven without the host: ten steps captured in a graph, dt on the device
        step_case("graph 32^3 x10", (32, 32, 32), steps=10, mach=0.2, kind="graph"),
        # the reference's published run: its cell64 deck, 100 steps from the CGS initial state
        {"name": "deck 64^3 x100", "kind": "deck", "nx": 64, "ny": 64, "nz": 64, "steps": 100},
        # odd extents: ragged tiles in every direction, rows that end inside a 16-byte pair
        step_case("step 130x97x61", (130, 97, 61)),
        # an ordinary box, one of a request stream served one at a time
        step_case("step 128^3", (128, 128, 128)),
        # a large production box that one user runs alone
        step_case("step 256^3", (256, 256, 256)),
        # the benchmark's box: 512^3, 29 GB of state
        step_case("step 512^3", (512, 512, 512)),
        # a program that composes the step itself from the per-kernel calls, as the
        # reference's main loop does (fill, ctoprim with the Courant number, diffterm,
        # hypterm, update, three times)
        step_case("operators 200x180x160", (200, 180, 160), kind="operators"),
        # the reference's multi-box form: one periodic domain as 64 boxes, one dt
        {"name": "domain 256^3 of 64^3", "kind": "domain", "nb": 4, "m": 64, "mach": 0.085},
        # independent boxes of uneven edges advanced together, FP32 flux arithmetic
        {"name": "batch fp32 64 boxes x4", "kind": "batch", "boxes": 64, "lo": 16, "hi": 96, "listed_edges": True,
         "steps": 4, "fp32": True},
        # the same in FP64
        {"name": "batch fp64 64 boxes x4", "kind": "batch", "boxes": 64, "lo": 16, "hi": 96, "listed_edges": True,
         "steps": 4, "fp32": False},
        # a server's cycle on the request stream's sizes: admit boxes, set their targets, a
        # chunk of steps, status, results back, retire
        {"name": "serve fp32 40 boxes x8", "kind": "serve", "boxes": 40, "lo": 24, "hi": 128, "listed_edges": False,
         "steps": 8, "fp32": True},
    ]


def log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "graph", "deck", "operators", "domain", "batch", "batch", "serve"])
    mach = round(rng.uniform(0.05, 0.3), 3)
    if kind == "step" or kind == "operators":
        # cubes and bricks of 8..512 cells a side
        if rng.random() < 0.4:
            e = log_int(rng, 12, 400 if kind == "step" else 256)
            n = (e, e, e)
        else:
            n = [log_int(rng, 8, 512 if kind == "step" else 256) for _ in range(3)]
        return {k: v for k, v in step_case("", n, mach=mach, kind=kind).items() if k != "name"}
    if kind == "graph":
        n = [log_int(rng, 12, 96) for _ in range(3)]
        return {k: v for k, v in step_case("", n, steps=rng.randint(2, 10), mach=mach, kind=kind).items() if k != "name"}
    if kind == "deck":
        e = rng.choice([16, 24, 32, 40, 48, 64])
        return {"kind": "deck", "nx": e, "ny": e, "nz": e, "steps": rng.randint(20, 100)}
    if kind == "domain":
        m = rng.choice([16, 24, 32, 40, 48, 64, 80])
        return {"kind": "domain", "nb": rng.randint(2, 4), "m": m, "mach": mach}
    if kind == "batch":
        return {"kind": "batch", "boxes": rng.randint(8, 64), "lo": rng.randint(8, 32), "hi": rng.randint(48, 112),
                "listed_edges": False, "steps": rng.randint(2, 6), "fp32": rng.random() < 0.5}
    return {"kind": "serve", "boxes": rng.randint(8, 40), "lo": 24, "hi": rng.randint(64, 128), "listed_edges": False,
            "steps": rng.randint(4, 8), "fp32": rng.random() < 0.7}


# ----------------------------------------------------------------------- inputs
def waves(n, rng, kmax=2, nmodes=4):
    """A seeded sum of products of sines over wavenumbers 1..kmax, scaled to 1, [nz, ny, nx]."""
    out = torch.zeros((n[2], n[1], n[0]), dtype=torch.float64, device="cuda")
    x = [(torch.arange(v, dtype=torch.float64, device="cuda") + 0.5) * (2 * math.pi / v) for v in n]
    for _ in range(nmodes):
        k = rng.integers(1, kmax + 1, size=3)
        ph = rng.uniform(0.0, 2.0 * math.pi, size=3)
        f = [torch.sin(int(k[d]) * x[d] + float(ph[d])) for d in range(3)]
        out.addcmul_(f[2][:, None, None] * float(rng.uniform(0.5, 1.0)), f[1][None, :, None] * f[0][None, None, :])
    return out.div_(out.abs().max())


def flow(n, seed, mach):
    """Conserved state [5, nz, ny, nx] of a smooth low-Mach flow (rho, p = 1 +- 5 %)."""
    rng = np.random.default_rng(seed)
    c0 = math.sqrt(GAMMA)
    rho = waves(n, rng).mul_(0.05).add_(1.0)
    u, v, w = (waves(n, rng).mul_(mach * c0) for _ in range(3))
    p = waves(n, rng).mul_(0.05).add_(1.0)
    return torch.stack([rho, rho * u, rho * v, rho * w, p / (GAMMA - 1.0) + 0.5 * rho * (u * u + v * v + w * w)])


def cgs_flow(n, seed):
    """The CGS initial state of the reference's cell32 and cell64 decks (rho 1e-3, |u| 1e4,
    e 2.5e9), its velocities scaled and shifted by the seed."""
    rng = np.random.default_rng(seed)
    amp, ph = rng.uniform(0.8, 1.0, size=3), rng.uniform(0.0, 2.0 * math.pi, size=3)
    x, y, z = (torch.arange(n[d], dtype=torch.float64, device="cuda") * (2 * math.pi / n[d]) + float(ph[d])
               for d in range(3))
    z, y, x = z[:, None, None], y[None, :, None], x[None, None, :]
    u = 1.1e4 * float(amp[0]) * torch.sin(x) * torch.sin(2 * y) * torch.sin(3 * z)
    v = 1.0e4 * float(amp[1]) * torch.sin(2 * x) * torch.sin(4 * y) * torch.sin(z)
    w = 1.2e4 * float(amp[2]) * torch.sin(3 * x) * torch.cos(2 * y) * torch.sin(2 * z)
    rho = 1.0e-3 + 1.0e-5 * torch.sin(x) * torch.cos(2 * y) * torch.cos(3 * z)
    e = 2.5e9 + 1.0e-3 * torch.sin(2 * x) * torch.cos(2 * y) * torch.sin(2 * z)
    return torch.stack([rho, rho * u, rho * v, rho * w, rho * (e + (u * u + v * v + w * w) / 2)])


def box_edges(case, seed):
    """Edges and Mach numbers of a batch (drawn by the case alone: another seed gives other
    states in boxes of the same sizes)."""
    rng = np.random.default_rng([case["boxes"], case["lo"], case["hi"]])
    if case["listed_edges"]:
        edges = rng.choice((16, 24, 32, 48, 64, 96), case["boxes"])
    else:
        edges = rng.integers(case["lo"], case["hi"] + 1, case["boxes"])
    return [int(e) for e in edges], rng.uniform(0.05, 0.3, case["boxes"])


def box_states(case, seed):
    edges, machs = box_edges(case, seed)
    return [(e, flow((e, e, e), [seed, i], float(m))) for i, (e, m) in enumerate(zip(edges, machs))]


def extents(case):
    return (case["nx"], case["ny"], case["nz"])


def spacing(n):
    return tuple(SIDE / v for v in n)


# ----------------------------------------------------------------------- the passes
class State:
    pass


def prepare(case, seed):
    s = State()
    s.case, s.kind = case, case["kind"]
    if s.kind in ("step", "graph", "deck", "operators"):
        n = extents(case)
        s.lay = lay = BoxLayout(n)
        s.dx = spacing(n)
        s.cfl = cfl_of(max(n))
        s.arrays = ops.allocate_variables(lay)
        g = lay.dimg
        U = s.arrays[0].view(NC, g[2], g[1], lay.xg)[:, NG:NG + n[2], NG:NG + n[1], NG:NG + n[0]]
        U.copy_(cgs_flow(n, seed) if s.kind == "deck" else flow(n, seed, case["mach"]))
        if s.kind != "operators":
            s.stepper = ops.Stepper(lay, s.dx, s.cfl, ETA, ALAM)
        if s.kind == "deck":
            s.start = s.arrays[0].clone()
        if s.kind == "graph":
            start = s.arrays[0].clone()
            s.dt = torch.zeros(1, dtype=torch.float64, device="cuda")
            s.stepper.advance_async(*s.arrays, s.dt)
            s.arrays[0].copy_(start)
            torch.cuda.synchronize()
            s.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s.graph):
                for _ in range(case["steps"]):
                    s.stepper.advance_async(*s.arrays, s.dt)
    elif s.kind == "domain":
        n = (case["nb"] * case["m"],) * 3
        s.domain = domain.Domain(n, case["m"], spacing(n), cfl_of(n[0]), ETA, ALAM)
        s.arrays = s.domain.allocate()
        s.domain.scatter(flow(n, seed, case["mach"]), NC, s.arrays[0])
    else:
        s.boxes = [(e, u.reshape(-1)) for e, u in box_states(case, seed)]
        room = sum(batch.box_bytes(e, case["fp32"]) for e, _ in s.boxes) + (16 << 20)
        s.engine = batch.BatchEngine(room, fp32=case["fp32"], max_boxes=len(s.boxes))
        s.out = torch.empty(sum(u.numel() for _, u in s.boxes), dtype=torch.float64, device="cuda")
        if s.kind == "batch":
            s.ids = [s.engine.add(u, e) for e, u in s.boxes]
    return s


def run(s):
    return PASSES[s.kind](s)


def run_step(s):
    for _ in range(s.case["steps"]):
        dt = s.stepper.new_advance(*s.arrays)
    return step_outputs(s.arrays, dt)


def run_graph(s):
    s.graph.replay()
    return step_outputs(s.arrays, s.dt)


def run_deck(s):
    s.arrays[0].copy_(s.start)
    return run_step(s)


def run_operators(s):
    lay, dx = s.lay, s.dx
    lo, hi = lay.lo, lay.hi
    U, Unew, Q, D, F = s.arrays
    for phase, X in ((1, U), (2, Unew), (3, Unew)):
        ops.fill_boundary(X, lay.n, lay.dimg)
        if phase == 1:
            dt = s.cfl / ops.ctoprim(lo, hi, X, Q, dx, NG, 1.0e-50)
        else:
            ops.ctoprim(lo, hi, X, Q, dx, NG)
        ops.diffterm(lo, hi, NG, dx, Q, D, ETA, ALAM)
        ops.hypterm(lo, hi, NG, dx, X, Q, F)
        ops.rk_update(phase, lo, hi, NG, U, Unew, D, F, dt)
    return step_outputs(s.arrays, dt)


def run_domain(s):
    dt = s.domain.advance(*s.arrays)
    return step_outputs(s.arrays, dt)


def step_outputs(arrays, dt):
    return dict(zip(("U", "Unew", "Q", "D", "F"), arrays), dt=dt)


def run_batch(s):
    s.engine.step(s.case["steps"])
    return collect(s, s.ids)


def run_serve(s):
    ids = [s.engine.add(u, e) for e, u in s.boxes]
    for i in ids:
        s.engine.set_target(i, s.case["steps"])
    s.engine.step(s.case["steps"])
    got = collect(s, ids)
    for i in ids:
        s.engine.remove(i)
    return got


def collect(s, ids):
    q = s.engine.query(ids)
    at = 0
    for i, (_, u) in zip(ids, s.boxes):
        s.engine.read(i, s.out[at:at + u.numel()])
        at += u.numel()
    return {"U": s.out, "dt": np.array([q[i]["dt"] for i in ids])}


PASSES = {"step": run_step, "graph": run_graph, "deck": run_deck, "operators": run_operators, "domain": run_domain,
          "batch": run_batch, "serve": run_serve}


def work(case):
    """Per step, the state is read once and every array the step leaves is written once
    (U, Unew, Q over their ghosts; D, F); a batched box has its U alone."""
    kind = case["kind"]
    if kind in ("batch", "serve"):
        edges, _ = box_edges(case, 0)
        cells = sum(e ** 3 for e in edges)
        # resident: U in and out each step, U out to the caller; served: U in from the caller too
        bytes_ = 8 * 5 * cells * (2 * case["steps"] + (2 if kind == "batch" else 4))
        return {"bytes": bytes_, "flops": 3 * STAGE_FLOPS * cells * case["steps"]}
    n = (case["m"],) * 3 if kind == "domain" else extents(case)
    boxes = case["nb"] ** 3 if kind == "domain" else 1
    steps = case.get("steps", 1)
    c = n[0] * n[1] * n[2] * boxes
    g = (n[0] + 8) * (n[1] + 8) * (n[2] + 8) * boxes
    return {"bytes": 8 * steps * (5 * c + 16 * g + 10 * c), "flops": 3 * STAGE_FLOPS * c * steps}


# ----------------------------------------------------------------------- plain torch
AXIS = (2, 1, 0)  # dimension of x, y, z in [nz, ny, nx]


def first(f, d, h):
    """8th-order first derivative along axis d of a periodic field."""
    a = AXIS[d]
    return sum(c * (f.roll(-m, a) - f.roll(m, a)) for m, c in enumerate(FIRST, 1)) / h


def second(f, d, h):
    a = AXIS[d]
    return (SECOND[0] * f + sum(c * (f.roll(-m, a) + f.roll(m, a)) for m, c in enumerate(SECOND[1:], 1))) / (h * h)


def primitives(U):
    rho = U[0]
    u, v, w = U[1] / rho, U[2] / rho, U[3] / rho
    e = U[4] / rho - 0.5 * (u * u + v * v + w * w)
    return [rho, u, v, w, (GAMMA - 1.0) * e * rho, e / CV]


def divergence(U, q, dx):
    """hypterm: minus the divergence of the inviscid fluxes."""
    F = [torch.zeros_like(U[0]) for _ in range(5)]
    for d in range(3):
        vel, p = q[1 + d], q[4]
        F[0] -= first(U[1 + d], d, dx[d])
        for l in range(3):
            F[1 + l] -= first(U[1 + l] * vel + p if l == d else U[1 + l] * vel, d, dx[d])
        F[4] -= first((U[4] + p) * vel, d, dx[d])
    return torch.stack(F)


def diffusion(q, dx, eta=ETA, alam=ALAM):
    """diffterm: the viscous stresses' divergence, heat conduction and mechanical work."""
    vel, T = q[1:4], q[5]
    same = [first(vel[d], d, dx[d]) for d in range(3)]  # ux, vy, wz
    D = [torch.zeros_like(T)]
    for l in range(3):
        s = sum((4.0 / 3.0 if d == l else 1.0) * second(vel[l], d, dx[d]) for d in range(3))
        s = s + sum(first(same[d], l, dx[l]) for d in range(3) if d != l) / 3.0
        D.append(eta * s)
    div = 2.0 / 3.0 * (same[0] + same[1] + same[2])
    mech = sum((2.0 * same[d] - div) * same[d] for d in range(3))
    for a, b in ((0, 1), (0, 2), (1, 2)):
        tau = first(vel[a], b, dx[b]) + first(vel[b], a, dx[a])
        mech = mech + tau * tau
    heat = alam * sum(second(T, d, dx[d]) for d in range(3))
    D.append(heat + eta * mech + sum(D[1 + l] * vel[l] for l in range(3)))
    return torch.stack(D)


def rk3(U, dx, cfl):
    """One step from interior state U: (U, U of stage 2/3, its primitives, D, F, dt)."""
    q = primitives(U)
    c = torch.sqrt(GAMMA * q[4] / q[0])
    dt = cfl / max(float(((c + q[1 + d].abs()) / dx[d]).max()) for d in range(3))
    del c
    A = U
    for base, new in ((0.0, 1.0), (0.75, 0.25), (1.0 / 3.0, 2.0 / 3.0)):
        if base:
            q = primitives(A)
        before = A
        D, F = diffusion(q, dx), divergence(A, q, dx)
        A = base * U + new * (A + dt * (D + F))
    return A, before, torch.stack(q), D, F, dt


def ghosted(f, n, boxes=None):
    """Interior [ncomp, nz, ny, nx] of the whole domain -> flat ghosted arrays of its boxes."""
    N = f.shape[:0:-1]
    nb = [N[d] // n[d] for d in range(3)]
    xg = -(-(n[0] + 2 * NG) // 16) * 16
    out = torch.zeros((nb[0] * nb[1] * nb[2], f.shape[0], n[2] + 2 * NG, n[1] + 2 * NG, xg), dtype=torch.float64,
                      device=f.device)
    for b in range(out.shape[0]):
        at = (b % nb[0], (b // nb[0]) % nb[1], b // (nb[0] * nb[1]))
        ix = [(torch.arange(n[d] + 2 * NG, device=f.device) - NG + at[d] * n[d]) % N[d] for d in range(3)]
        for l in range(f.shape[0]):
            out[b, l, :, :, :n[0] + 2 * NG] = f[l][ix[2]][:, ix[1]][:, :, ix[0]]
    return out.reshape(-1)


def unghosted(f, n):
    """The same for arrays without ghosts."""
    N = f.shape[:0:-1]
    nb = [N[d] // n[d] for d in range(3)]
    x = -(-n[0] // 16) * 16
    out = torch.zeros((nb[0] * nb[1] * nb[2], f.shape[0], n[2], n[1], x), dtype=torch.float64, device=f.device)
    for b in range(out.shape[0]):
        i, j, k = (b % nb[0]) * n[0], ((b // nb[0]) % nb[1]) * n[1], b // (nb[0] * nb[1]) * n[2]
        out[b, :, :, :, :n[0]] = f[:, k:k + n[2], j:j + n[1], i:i + n[0]]
    return out.reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("batch", "serve"):
        states, dts = [], []
        for e, U in box_states(case, seed):
            for _ in range(case["steps"]):
                U, _, _, _, _, dt = rk3(U, (SIDE / e,) * 3, 0.5)
            # the engine's dt is that of the next step once a step has ended
            q = primitives(U)
            c = torch.sqrt(GAMMA * q[4] / q[0])
            dts.append(0.5 / (float(max((c + q[1 + d].abs()).max() for d in range(3))) * e / SIDE))
            states.append(U.reshape(-1))
        return {"U": torch.cat(states), "dt": np.array(dts)}
    if kind == "domain":
        n = (case["m"],) * 3
        N = (case["nb"] * case["m"],) * 3
        U = flow(N, seed, case["mach"])
    else:
        n = N = extents(case)
        U = cgs_flow(n, seed) if kind == "deck" else flow(n, seed, case["mach"])
    for _ in range(case.get("steps", 1)):
        before = U  # the ghosts of U are images of the step's own start
        U, Unew, q, D, F, dt = rk3(U, spacing(N), cfl_of(max(N)))
    out = {"Unew": ghosted(Unew, n), "Q": ghosted(q, n), "D": unghosted(D, n), "F": unghosted(F, n), "dt": dt}
    del Unew, q, D, F
    whole = ghosted(before, n).view(-1, NC, n[2] + 2 * NG, n[1] + 2 * NG, -(-(n[0] + 2 * NG) // 16) * 16)
    inner = unghosted(U, n).view(-1, NC, n[2], n[1], -(-n[0] // 16) * 16)
    whole[:, :, NG:NG + n[2], NG:NG + n[1], NG:NG + n[0]] = inner[..., :n[0]]
    out["U"] = whole.reshape(-1)
    return out
