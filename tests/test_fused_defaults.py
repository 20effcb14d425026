"""The fused pass's default configuration in FP64: wide blocks with strips (code 9) at N = 3 * 2^k beyond the last-level
cache and at no other size of that range.  (A handle without GW sourcing is not tuned: its tune() returns the default.)"""
import pytest

from axion_grav_amd import capi
from tests.conftest import SQ_HALF, phys


@pytest.mark.gpu
@pytest.mark.parametrize("N,code", [(48, 0), (96, 0), (144, 0), (192, 9), (216, 0), (288, 0), (324, 0), (384, 9), (432, 0)])
def test_wide_blocks(N, code):
    print("[case] fused default", N, flush=True)
    with capi.Lattice(capi.make_params(N, phys(N)["dspa"], SQ_HALF, grav_spec=False, spec_est=False)) as L:
        assert L.tune()[0] == code
