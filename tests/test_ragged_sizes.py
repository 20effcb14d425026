"""Lattices whose size has two to four factors of three and at least three of two (the compile-time engine's
radix-9 and radix-3 passes): the step against the oracle, and above the oracle's sizes the GW spectrum
of one kick against 64-bit torch transforms of the same field."""
import numpy as np
import pytest

import oracle as O
from axion_grav_amd import capi
from tests.conftest import SQ_HALF, phys

pytestmark = pytest.mark.gpu


# 72 = 9 * 8, 144 = 9 * 16 and 216 = 27 * 8 take each kind of pass; dspa = 0.3 has no exact reciprocal.  FP64:
# the bar of the GW parity tests; FP32: 2^-24 for each of the transform's log2(N^3) < 24 stages.
@pytest.mark.parametrize("N,dspa,fix,prec,tol", [
    (72, 0.3, False, capi.FP64, 1e-10), (72, 0.25, True, capi.FP32C, 3e-6), (144, 0.25, False, capi.FP64, 1e-10),
    (144, 0.3, False, capi.FP32, 3e-6), (216, 0.25, True, capi.FP64, 1e-10), (216, 0.25, False, capi.FP32C, 3e-6)])
def test_step_matches_oracle(N, dspa, fix, prec, tol):
    print("[case] ragged", N, dspa, fix, prec, flush=True)
    P = dict(phys(N), dspa=dspa, dwav=2 * 3.14159265359 / dspa / N, dv_spa=dspa ** 3)
    phi, pi = O.ic_flat(N, 5, 1.5, P["dwav"])
    steps = 2 if N < 200 else 1
    with capi.Lattice(capi.make_params(N, dspa, SQ_HALF, precision=prec, gw_fix_swap=fix)) as L:
        L.set_fields(phi, pi)
        L.advance_steps(1.0, 0.02, steps)
        A = L.gw_state()
        g_phi, g_pi = L.get_fields()
    OA = O.new_gw_state(N)
    O.symplectic(phi, pi, OA, 1.0, 0.02, steps, P, fix_swap=fix)
    if prec == capi.FP64:
        assert np.array_equal(g_phi, phi) and np.array_equal(g_pi, pi)
    for m in range(4):
        ref = OA[m][:, :, : N // 2 + 1]
        assert np.abs(A[m] - ref).max() <= tol * np.abs(ref).max(), m


def kick_numer(phi, dspa, tau, dt, nb):
    """numer per bin after one kick of a field at rest, in torch: |A|^2 summed over the shells."""
    import torch

    n = phi.shape[0]
    w = torch.arange(n)
    w = torch.where(w < n // 2, w, w - n).double()
    dwav = 2 * 3.14159265359 / dspa / n
    nz, ny, nx = w[:, None, None], w[None, :, None], w[: n // 2 + 1][None, None, :]
    rho2 = nx * nx + ny * ny + 0 * nz
    q = torch.sqrt(rho2 + nz * nz)
    q[0, 0, 0] = 1
    rho = torch.sqrt(rho2)
    on = rho > 0
    c, s = torch.where(on, nx / torch.where(on, rho, 1), 1), torch.where(on, ny / torch.where(on, rho, 1), 0)
    p = [torch.complex(nz / q * c, -s), torch.complex(nz / q * s, c), torch.complex(-rho / q, 0 * q)]
    grad = [(torch.roll(phi, -1, a) - torch.roll(phi, 1, a)) / (2 * dspa) for a in (2, 1, 0)]
    sp = sn = 0
    for i in range(3):
        for j in range(i + 1):
            d = torch.conj(torch.fft.rfftn(2 * (grad[i] * torch.conj(grad[j])).real))
            pol = p[i] * p[j] * (0.5 if i == j else 1.0)
            sp, sn = sp + pol * d, sn + torch.conj(pol) * d
    co, si = torch.cos(q * dwav * tau), torch.sin(q * dwav * tau)
    dw = tau * dt * dspa ** 3 * 0.5
    a12 = dw * (si * sp + co * sn)
    power = (dw * co * sp).abs() ** 2 + (dw * si * sn).abs() ** 2 + a12.abs() ** 2 + \
        (a12 - dw * co * (rho2 / q ** 2 / 2) * d).abs() ** 2
    power[0, 0, 0] = 0
    wt = torch.full((n // 2 + 1,), 2.0, dtype=torch.float64)
    wt[0] = wt[-1] = 1
    n2 = torch.round(rho2 + nz * nz).long().numpy()
    tab = np.floor(np.sqrt(np.arange(n2.max() + 1.0)) * dwav / (3.14159265359 / dspa / nb) + 0.5 + 0.5).astype(np.int64)
    b = torch.from_numpy(np.where((tab >= 1) & (tab <= nb), tab - 1, nb)[n2])
    return torch.zeros(nb + 1, dtype=torch.float64).index_add(0, b.reshape(-1), (power * wt).reshape(-1))[:nb]


# FP64: 1e-12 of each bin, some ten stages of 2^-53 over sums of like terms; FP32: a mode's relative error
# of 3e-6 doubles in its square
@pytest.mark.parametrize("N,prec,tol", [(288, capi.FP64, 1e-12), (432, capi.FP32C, 6e-6), (648, capi.FP64, 1e-12)])
def test_kick_spectrum_matches_torch(N, prec, tol):
    import torch

    print("[case] ragged spectrum", N, prec, flush=True)
    nb, dspa, dt = 32, 0.25, 0.02
    with capi.Lattice(capi.make_params(N, dspa, SQ_HALF, precision=prec, num_bin_grav=nb)) as L:
        L.init_flat(9, 2.0)
        phi, _ = L.get_fields()
        L.advance_steps(1.0, dt, 1)
        s = L.gw_spectrum()
    ref = kick_numer(torch.from_numpy(phi), dspa, 1.0 + dt / 2, dt, nb).numpy()
    assert np.all(np.isfinite(s["numer"]))
    # the sources of |k| < 2 fields reach |k| < 4 of pi / dspa = 12.6: the bins below that hold the signal
    k = np.arange(nb) < nb // 4
    assert np.all(np.abs(s["numer"] - ref)[k] <= tol * ref[k]), np.abs(s["numer"] / ref - 1)[k].max()
