"""Passes that the other tests reach at other sizes only: the fused pass's and the y pass's configurations, the tuner and
the adjoint at the sizes with two or more factors of three, the radix-9 columns of the two-column y pass and
the z pass's narrow tiles from 576, the stacked y pass at 768, and the default blocks at 192 in FP64.  The
bars are those of the tests that they call."""
import numpy as np
import pytest

import tests.test_adjoint as adjoint
import tests.test_gpu_parity as parity
import tests.test_ragged_sizes as ragged
from axion_grav_amd import capi
from tests.conftest import SQ_HALF, phys

pytestmark = pytest.mark.gpu


def run(N, prec, steps=3):
    with capi.Lattice(capi.make_params(N, phys(N)["dspa"], SQ_HALF, precision=prec, num_bin_grav=32)) as L:
        L.init_flat(11, 2.0)
        L.advance_steps(1.0, 0.05, steps)
        return (*L.get_fields(), *L.gw_state())


# every site is updated once whatever the block order: the same bits.  72 has six rows a block, twelve in the wide
# one; 216 and 288 two and one (four and three), 288 with 4.5 waves
@pytest.mark.parametrize("N,prec", [(72, capi.FP64), (72, capi.FP32C), (144, capi.FP32), (192, capi.FP64), (216, capi.FP64),
                                    (288, capi.FP32C)])
def test_fused_configurations_bit_identical(N, prec, monkeypatch):
    print("[case] fused configurations", N, prec, flush=True)
    ref = run(N, prec)
    for v in (0, 1, 4, 5, 8, 9, 12, 13):
        monkeypatch.setenv("AXG_KICK_VARIANT", str(v))
        for a, b in zip(run(N, prec), ref):
            assert np.array_equal(a, b), v


@pytest.mark.parametrize("N,prec", [(72, capi.FP64), (144, capi.FP32C)])
def test_ypass_and_tuner(N, prec, monkeypatch):
    parity.test_ypass_variants_bit_identical(N, prec, monkeypatch)
    monkeypatch.delenv("AXG_YPASS_VARIANT")
    parity.test_tune_keeps_fields_and_results(prec, N)


@pytest.mark.parametrize("N,prec", [(576, capi.FP64), (576, capi.FP32C), (648, capi.FP32), (864, capi.FP32C)])
def test_ypass_line_tiles_radix9(N, prec, monkeypatch):
    parity.test_ypass_line_tiles_large(N, prec, monkeypatch)


@pytest.mark.parametrize("N,prec,tol", [(576, capi.FP32C, 6e-6), (576, capi.FP64, 1e-12), (648, capi.FP32, 6e-6)])
def test_kick_spectrum(N, prec, tol):
    ragged.test_kick_spectrum_matches_torch(N, prec, tol)


def test_largest_radix9_lattice():
    parity.test_largest_lattices_fp32c_tracks_fp64(864)


@pytest.mark.parametrize("prec,N,K,fix,tol", [("fp64", 72, 5, False, 1e-7), ("fp64", 72, 4, True, 1e-7), ("fp32c", 72, 5, True, 2e-4),
                                              ("fp32c", 72, 4, False, 2e-4), ("fp32c", 36, 5, True, 2e-4), ("fp32c", 36, 4, False, 2e-4)])
def test_gradient(prec, N, K, fix, tol):
    adjoint.test_gpu_gradient_matches_oracle(prec, N, K, fix, tol, "phys")


def test_stacked_y_pass_768():
    print("[case] stacked 768", flush=True)
    prm = capi.make_params(768, phys(768)["dspa"], SQ_HALF, precision=capi.FP32C, num_bin_grav=64)
    out = []
    for batch in (False, True):
        with capi.Lattice(prm) as L:
            L.init_flat(3, 1.0)
            if batch:
                capi.batch_advance([L], 1.0, 0.05, 4, 2)
            else:
                L.advance_steps(1.0, 0.05, 4)
            out.append((L.gw_spectrum()["numer"], L.energy(1.2)))
    assert np.any(out[0][0] > 0) and np.all(np.isfinite(out[0][0]))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
