"""The field spectrum and covariance at the sizes without compile-time kernels, whose rows the binning folds itself: one
to three values a lane, and the smallest size."""
import pytest

import tests.test_spectrum_passes as passes
from axion_grav_amd import capi


@pytest.mark.gpu
@pytest.mark.parametrize("N,nb,prec,stream", [(8, 3, capi.FP64, None), (18, 6, capi.FP32C, None), (54, 12, capi.FP64, (3, 4, 77)),
                                              (108, 12, capi.FP32, None), (162, 12, capi.FP64, None), (324, 16, capi.FP32C, None)])
def test_spectrum_and_covariance(N, nb, prec, stream):
    passes.test_spectrum_and_covariance(N, nb, prec, stream)
