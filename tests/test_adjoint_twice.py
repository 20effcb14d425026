"""The adjoint fields read several times after a gradient, each alone and both together."""
import numpy as np
import pytest

from axion_grav_amd import capi
from tests.conftest import SQ_HALF
from tests.test_adjoint import CASE, fields, oparams


@pytest.mark.gpu
@pytest.mark.parametrize("N", [16, 108])
def test_adjoint_read_again(N):
    print("[case] adjoint read again", N, flush=True)
    c = CASE
    prm = capi.make_params(N, oparams(N, 1e-3)["dspa"], SQ_HALF, num_bin_grav=c["nb"], potential_kappa0=1e-3)
    with capi.Lattice(prm) as L:
        L.set_fields(*fields(N))
        for _ in range(2):
            f = L.get_fields()
            L.gradient(c["t1"], c["dt"], 3, 2, c["qlo"], c["qhi"])
            L.set_fields(*f)
            a, b = L.adjoint()
            assert np.abs(a).max() > 0 and np.abs(b).max() > 0
            n3, x, y = N ** 3, np.zeros_like(a), np.zeros_like(b)
            assert capi.lib().axg_get_adjoint(L._h, capi._ptr(x), None, n3) == 0
            assert capi.lib().axg_get_adjoint(L._h, None, capi._ptr(y), n3) == 0
            assert np.array_equal(x, a) and np.array_equal(y, b)
            L.gradient(c["t1"], c["dt"], 3, 2, c["qlo"], c["qhi"])
            L.set_fields(*f)
            assert capi.lib().axg_get_adjoint(L._h, None, capi._ptr(y), n3) == 0
            assert np.array_equal(y, b) and np.array_equal(L.adjoint()[0], a)
