"""The field spectrum's fused transforms at a size of each kind of engine (2^k, 3 * 2^k, 9 * 2^k, the runtime
plan) against the oracle: spectrum and covariance, with Philox draws and with the reference's stream,
whose draws a thread steps through."""
import numpy as np
import pytest

import oracle as O
from axion_grav_amd import capi
from tests.conftest import SQ_HALF, phys
from tests.test_gpu_parity import packed, relerr

pytestmark = pytest.mark.gpu


# the bars of the field spectrum's and the covariance's parity tests (tests/test_gpu_parity.py); FP32C fields
# are read back, so that both sides take the same values
@pytest.mark.parametrize("N,nb,prec,stream", [(24, 8, capi.FP64, (3, 4, 77)), (36, 8, capi.FP64, (3, 4, 77)), (36, 8, capi.FP64, None),
                                              (64, 12, capi.FP64, (7, 9, 1001)), (64, 12, capi.FP32, None),
                                              (72, 12, capi.FP64, None), (72, 12, capi.FP32C, (7, 9, 10 ** 9))])
def test_spectrum_and_covariance(N, nb, prec, stream):
    print("[case] spectrum passes", N, nb, prec, stream, flush=True)
    P = phys(N)
    phi, _ = O.ic_flat(N, 31, 2.0, P["dwav"])
    rng = np.random.default_rng(1)
    pi = rng.standard_normal((N, N, N)) + 1j * rng.standard_normal((N, N, N))
    with capi.Lattice(capi.make_params(N, P["dspa"], SQ_HALF, precision=prec, num_bin=nb, grav_spec=False)) as L:
        L.set_fields(phi, pi)
        phi, pi = L.get_fields()
        if stream:
            L.set_stream(*stream)
        L.defects()
        s = L.field_spectrum(3.0)
        cov, it = L.field_covariance(5, 3, 4, 0.0)
        if stream:
            assert L.stream_position() == stream[2] + 4 * 4 * N ** 3
    flags, _ = O.classify(phi)
    pw, num = O.conv_spectrum(pi, flags, nb, P["dspa"], P["dwav"], P["dv_spa"], P["dv_wav"])
    assert np.array_equal(s["num"], num) and relerr(s["conv"], pw * 9.0) < 1e-10
    tab = O.init_spectrum(nb, P["dspa"])
    _, inv, info = O.matrix_deconv(flags, nb, P["dwav"], P["dv_spa"], P["dv_wav"], tab)
    M = O.sym_from_packed(inv, nb) / np.outer(num, num)
    assert info == 0 and relerr(s["power"], M @ (pw * 9.0)) < 1e-8
    kw = {"stream": stream} if stream else {}
    ocov, oit, _ = O.field_covariance(flags, nb, P["dspa"], P["dwav"], s["power"], packed(M), 5, 3, 4, 0.0, **kw)
    assert it == oit == -5
    assert np.all(np.isfinite(ocov)) and relerr(cov, ocov) < 1e-6
