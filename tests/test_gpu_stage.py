"""The one-kernel RK stage (cns_stage.hip) where its 32 x 16 tiles and z runs end.

Every ABI array and dt after three steps must equal, bit for bit, the kernel-for-kernel
composition on the direct one-thread-per-cell kernels: both evaluate the same expressions
in the same order, so the tolerance is zero."""
import numpy as np
import pytest

from cns_nospec_amd import _lib, ops
from cns_nospec_amd.layout import BoxLayout
from cns_nospec_amd.state import sinusoid_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(31, 15, 4), (32, 16, 5), (33, 17, 9), (36, 31, 8), (65, 20, 30), (64, 64, 40),
                               (5, 130, 11), (200, 7, 6)])
def test_stage_kernel_equals_direct_kernels(device, n):
    import torch
    lay = BoxLayout(n)
    U0 = torch.from_numpy(sinusoid_state(lay, 17, mach=0.25, kmax=3)).to(device)
    got = {}
    for impl in (_lib.CNS_IMPL_TILED, _lib.CNS_IMPL_DIRECT):
        print(f"stage kernel n={n} impl={impl}", flush=True)
        ops.set_stencil_impl(impl)
        try:
            arrays = ops.allocate_variables(lay, device)
            arrays[0].copy_(U0)
            st = ops.Stepper(lay)
            st.set_fused(impl == _lib.CNS_IMPL_TILED)
            dts = [st.new_advance(*arrays) for _ in range(3)]
            got[impl] = (dts, [a.cpu().numpy() for a in arrays])
            st.close()
        finally:
            ops.set_stencil_impl(_lib.CNS_IMPL_TILED)
    (dts, arrays), (rdts, rarrays) = got[_lib.CNS_IMPL_TILED], got[_lib.CNS_IMPL_DIRECT]
    assert dts == rdts
    for a, b, name in zip(arrays, rarrays, ("U", "Unew", "Q", "D", "F")):
        assert np.array_equal(a, b), name


@pytest.mark.parametrize("first", ["stage", "direct", "unfused"])
def test_courant_maximum_does_not_outlive_a_step(device, first):
    """A step leaves its context's Courant maximum at zero on every route, so a slower flow
    stepped after a faster one, in any composition, gets its own dt."""
    import torch
    lay = BoxLayout((20, 18, 9))

    def fresh(mach):
        arrays = ops.allocate_variables(lay, device)
        arrays[0].copy_(torch.from_numpy(sinusoid_state(lay, 5, mach=mach, kmax=2)).to(device))
        return arrays

    def step(st, route, arrays):
        print(f"courant maximum route={route}", flush=True)
        ops.set_stencil_impl(_lib.CNS_IMPL_DIRECT if route == "direct" else _lib.CNS_IMPL_TILED)
        st.set_fused(route != "unfused")
        try:
            return st.new_advance(*arrays)
        finally:
            ops.set_stencil_impl(_lib.CNS_IMPL_TILED)

    ref = ops.Stepper(lay)
    want_fast, want_slow = ref.new_advance(*fresh(0.9)), ref.new_advance(*fresh(0.01))
    ref.close()
    alone = ops.Stepper(lay)
    assert alone.new_advance(*fresh(0.01)) == want_slow and want_slow > want_fast
    alone.close()

    st = ops.Stepper(lay)
    for route in (first, "stage", "direct", "unfused", "stage"):
        assert step(st, route, fresh(0.9)) == want_fast
        assert step(st, "stage", fresh(0.01)) == want_slow
        assert step(st, first, fresh(0.9)) == want_fast
        assert step(st, route, fresh(0.01)) == want_slow
    st.close()


def test_many_contexts_and_a_first_step_that_is_captured(device):
    """A context clears its Courant maximum with its first step, also when that one goes into a
    graph that never runs, and more contexts than the pinned page has slots return their own dt."""
    import torch
    lay = BoxLayout((8, 6, 5))

    def fresh(mach):
        arrays = ops.allocate_variables(lay, device)
        arrays[0].copy_(torch.from_numpy(sinusoid_state(lay, 5, mach=mach, kmax=2)).to(device))
        return arrays

    ref = ops.Stepper(lay)
    want = {mach: ref.new_advance(*fresh(mach)) for mach in (0.9, 0.01)}
    many = [ops.Stepper(lay) for _ in range(300)]
    for i in (0, 255, 256, 299):
        assert many[i].new_advance(*fresh(0.9)) == want[0.9]
        assert many[i].new_advance(*fresh(0.01)) == want[0.01]
    for st in many:
        st.close()
    st = ops.Stepper(lay)
    arrays, dt = fresh(0.9), torch.zeros(1, dtype=torch.float64, device=device)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        st.advance_async(*arrays, dt)
    del graph
    assert st.new_advance(*fresh(0.01)) == want[0.01]
    graph = torch.cuda.CUDAGraph()
    start = arrays[0].clone()
    with torch.cuda.graph(graph):
        st.advance_async(*arrays, dt)
    for _ in range(3):
        arrays[0].copy_(start)
        graph.replay()
        torch.cuda.synchronize()
        assert float(dt) == want[0.9]
        assert st.new_advance(*fresh(0.01)) == want[0.01]
    st.close()
    ref.close()


@pytest.mark.parametrize("n,separate", [((8, 8, 4096), True), ((4, 5, 4099), True), ((8, 8, 4095), False),
                                        ((9, 8, 4096), False), ((8, 9, 4096), False)])
def test_tall_columns_take_the_separate_kernels(device, n, separate):
    """Columns of up to 8 x 8 cells and at least 4096 planes are stepped kernel for kernel, their
    neighbours by the stage kernel; both to the bits of the direct kernels."""
    import torch
    lay = BoxLayout(n)
    U0 = torch.from_numpy(sinusoid_state(lay, 23, mach=0.2, kmax=2)).to(device)
    got = {}
    for impl in (_lib.CNS_IMPL_TILED, _lib.CNS_IMPL_DIRECT):
        print(f"tall column n={n} impl={impl}", flush=True)
        ops.set_stencil_impl(impl)
        try:
            arrays = ops.allocate_variables(lay, device)
            arrays[0].copy_(U0)
            st = ops.Stepper(lay)
            st.set_fused(impl == _lib.CNS_IMPL_TILED)
            st.profile(True)
            dts = [st.new_advance(*arrays) for _ in range(2)]
            kinds = {k for k, v in st.profile_read().items() if v[1] > 0}
            got[impl] = (dts, kinds, [a.cpu().numpy() for a in arrays])
            st.profile(False)
            st.close()
        finally:
            ops.set_stencil_impl(_lib.CNS_IMPL_TILED)
    (dts, kinds, arrays), (rdts, _, rarrays) = got[_lib.CNS_IMPL_TILED], got[_lib.CNS_IMPL_DIRECT]
    assert ("diffterm" in kinds) == separate and ("hypterm_rk" in kinds) != separate
    assert dts == rdts
    for a, b, name in zip(arrays, rarrays, ("U", "Unew", "Q", "D", "F")):
        assert np.array_equal(a, b), name
