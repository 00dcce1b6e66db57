"""The per-kernel calls where their tiles, z runs and planes end, bit for bit: the pipelined
stencils against the direct one-thread-per-cell kernels, the RK update against the same
expression in torch (one rounding per operation, as the library's)."""
import numpy as np
import pytest

from cns_nospec_amd import _lib, ops
from cns_nospec_amd.layout import NC, NG, BoxLayout
from cns_nospec_amd.state import ALAM, ETA, sinusoid_state

pytestmark = pytest.mark.gpu


# runs of one plane, of odd and even lengths; tiles that end in one column or row
@pytest.mark.parametrize("n", [(4, 4, 4), (20, 6, 5), (31, 7, 9), (33, 9, 31), (64, 8, 64), (65, 17, 130)])
def test_stencils_equal_direct_kernels(device, n):
    import torch
    lay = BoxLayout(n)
    dx = tuple(0.2 / v for v in n)
    U = torch.from_numpy(sinusoid_state(lay, 23, mach=0.25, kmax=3)).to(device)
    _, _, Q, _, _ = ops.allocate_variables(lay, device)
    ops.fill_boundary(U, lay.n, lay.dimg)
    ops.ctoprim(lay.lo, lay.hi, U, Q, dx, NG)
    got = []
    for impl in (_lib.CNS_IMPL_TILED, _lib.CNS_IMPL_DIRECT):
        print(f"operators n={n} impl={impl}", flush=True)
        _, _, _, D, F = ops.allocate_variables(lay, device)
        ops.set_stencil_impl(impl)
        try:
            ops.diffterm(lay.lo, lay.hi, NG, dx, Q, D, ETA, ALAM)
            ops.hypterm(lay.lo, lay.hi, NG, dx, U, Q, F)
        finally:
            ops.set_stencil_impl(_lib.CNS_IMPL_TILED)
        torch.cuda.synchronize()
        got.append((D.cpu().numpy(), F.cpu().numpy()))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("n", [(4, 4, 4), (17, 5, 6), (48, 33, 7), (130, 70, 60)])
@pytest.mark.parametrize("phase", [1, 2, 3])
def test_rk_update_equals_torch(device, n, phase):
    import torch
    lay = BoxLayout(n)
    rng = torch.Generator(device="cpu").manual_seed(31)
    U, Unew, _, D, F = (t.copy_(torch.rand(t.shape, generator=rng, dtype=torch.float64))
                        for t in ops.allocate_variables(lay, device))
    g = lay.dimg
    box = (slice(None), slice(NG, NG + n[2]), slice(NG, NG + n[1]), slice(NG, NG + n[0]))
    u0, w0 = U.clone(), Unew.clone()
    u, w = (t.view(NC, g[2], g[1], lay.xg)[box] for t in (u0, w0))
    x = -(-n[0] // 16) * 16
    d, f = (t.view(NC, n[2], n[1], x)[..., :n[0]] for t in (D, F))
    dt = 0.0137
    if phase == 1:
        w.copy_(u + dt * (d + f))
    elif phase == 2:
        w.copy_(0.75 * u + 0.25 * (w + dt * (d + f)))
    else:
        u.copy_(1.0 / 3.0 * u + 2.0 / 3.0 * (w + dt * (d + f)))
    print(f"rk_update n={n} phase={phase}", flush=True)
    ops.rk_update(phase, lay.lo, lay.hi, NG, U, Unew, D, F, dt)
    torch.cuda.synchronize()
    assert torch.equal(U, u0) and torch.equal(Unew, w0)


def test_fill_boundary_of_more_than_32_bits_of_ghost_cells(device):
    """A long thin box whose ghost cells do not fit 32 bits (2^32 + 1152 of them; 193 GB): every ghost
    cell holds its periodic image."""
    import torch
    torch.cuda.empty_cache()
    n = (1 << 25, 4, 4)
    lay = BoxLayout(n)
    if torch.cuda.mem_get_info()[0] < lay.ghosted_len(NC) * 8 + (4 << 30):
        pytest.skip("needs 198 GB of free GPU memory")
    g = lay.dimg
    U = torch.full((lay.ghosted_len(NC),), float("nan"), dtype=torch.float64, device=device)
    v = U.view(NC, g[2], g[1], lay.xg)
    x = torch.arange(n[0], dtype=torch.float64, device=device)
    rows = {}
    for l in range(NC):
        for k in range(n[2]):
            for j in range(n[1]):
                rows[l, k, j] = 1e8 * (1 + j + n[1] * (k + n[2] * l))
                torch.add(x, rows[l, k, j], out=v[l, NG + k, NG + j, NG:NG + n[0]])
    print("fill_boundary of 2^25 x 4 x 4", flush=True)
    ops.fill_boundary(U, lay.n, lay.dimg)
    torch.cuda.synchronize()
    want = torch.cat([x[-NG:], x, x[:NG]])
    for l in range(NC):
        for k in range(g[2]):
            for j in range(g[1]):
                assert torch.equal(v[l, k, j, :g[0]], want + rows[l, (k - NG) % n[2], (j - NG) % n[1]]), (l, k, j)
    del U, v, x, want
    torch.cuda.empty_cache()
