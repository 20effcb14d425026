"""The fused pass's default configuration in FP64: wide blocks with strips (code 9) at N = 3 * 2^k beyond the last-level
cache and at no other size of that range, and the same bits in a batch's stacks, which keep the narrow ones.  (A handle
without GW sourcing is not tuned: its tune() returns the default.)"""
import numpy as np
import pytest

from axion_grav_amd import capi
from tests.conftest import SQ_HALF, phys


@pytest.mark.gpu
@pytest.mark.parametrize("N,code", [(48, 0), (96, 0), (144, 0), (192, 9), (216, 0), (288, 0), (324, 0), (384, 9), (432, 0)])
def test_wide_blocks(N, code):
    print("[case] fused default", N, flush=True)
    with capi.Lattice(capi.make_params(N, phys(N)["dspa"], SQ_HALF, grav_spec=False, spec_est=False)) as L:
        assert L.tune()[0] == code


@pytest.mark.gpu
def test_stack_matches_single():
    print("[case] fused default in a stack", flush=True)
    prm = capi.make_params(192, phys(192)["dspa"], SQ_HALF, spec_est=False)
    with capi.Lattice(prm) as one, capi.Lattice(prm) as a, capi.Lattice(prm) as b:
        for L, seed in ((one, 1), (a, 1), (b, 2)):
            L.init_flat(seed, 1.0)
        one.advance_steps(1.0, 0.05, 4)
        capi.batch_advance([a, b], 1.0, 0.05, 4, 2)
        for x, y in zip((*one.get_fields(), *one.gw_state()), (*a.get_fields(), *a.gw_state())):
            assert np.array_equal(x, y)
