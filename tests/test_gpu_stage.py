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
