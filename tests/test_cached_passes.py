"""The passes of a single lattice with cached accesses (FP32 storage whose step stays in the last-level cache)
against the stacked launch of two such lattices, which streams: sizes on both sides of the rule's two bounds."""
import numpy as np
import pytest

from axion_grav_amd import capi
from tests.conftest import SQ_HALF, phys

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [capi.FP32C, capi.FP32])
@pytest.mark.parametrize("N,fix", [(64, False), (72, False), (72, True), (96, True), (128, False), (144, False)])
def test_single_matches_stack_bit_for_bit(N, fix, prec):
    print("[case] cached passes", N, fix, prec, flush=True)
    P = phys(N)
    par = dict(precision=prec, gw_fix_swap=fix)

    def made(seed):
        L = capi.Lattice(capi.make_params(N, P["dspa"], SQ_HALF, **par))
        L.init_flat(seed, 4.001 * P["dwav"])
        return L

    with made(1) as one, made(1) as a, made(2) as b:
        one.advance_steps(1.0, 0.05, 4)
        capi.batch_advance([a, b], 1.0, 0.05, 4, 2)
        for x, y in zip((*one.get_fields(), *one.gw_state()), (*a.get_fields(), *a.gw_state())):
            assert np.array_equal(x, y)
