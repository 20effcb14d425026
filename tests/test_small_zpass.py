"""The accumulation pass of the small lattices (six components transformed at once) against the oracle, at
every size and storage around the sizes where it takes over, in both index orders of the GW update."""
import numpy as np
import pytest

import oracle as O
from axion_grav_amd import capi
from tests.conftest import SQ_HALF, phys

pytestmark = pytest.mark.gpu


# FP64: the bar of the GW parity tests.  FP32: a transform of N^3 points rounds each of its log2(N^3)
# stages to 2^-24, about 6e-8 * 20 = 1.2e-6 of the largest mode at N = 128; two steps accumulate.
@pytest.mark.parametrize("prec,tol", [(capi.FP64, 1e-10), (capi.FP32C, 3e-6)])
@pytest.mark.parametrize("N,fix", [(16, True), (24, False), (32, True), (48, False), (64, True), (64, False), (96, False),
                                   (128, True)])
def test_accumulators_match_oracle(N, fix, prec, tol):
    print("[case] small z pass", N, fix, prec, flush=True)
    P = phys(N)
    phi, pi = O.ic_flat(N, 31, 4 * P["dwav"], P["dwav"])
    with capi.Lattice(capi.make_params(N, P["dspa"], SQ_HALF, precision=prec, gw_fix_swap=fix)) as L:
        L.set_fields(phi, pi)
        L.advance_steps(1.0, 0.05, 2)
        A = L.gw_state()
    OA = O.new_gw_state(N)
    O.symplectic(phi, pi, OA, 1.0, 0.05, 2, P, fix_swap=fix)
    for m in range(4):
        ref = OA[m][:, :, : N // 2 + 1]
        assert np.abs(A[m] - ref).max() <= tol * np.abs(ref).max(), m
