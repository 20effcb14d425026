"""Fields, flags and GW state through the pinned ring of the large host copies: byte-exact at sizes on both sides of
its least size, with a last chunk of every kind, into host memory at odd offsets, from two handles at once
and after the device's last handle gave the ring back."""
import ctypes as C
import threading

import numpy as np
import pytest

from axion_grav_amd import capi
from tests.conftest import SQ_HALF, phys

pytestmark = pytest.mark.gpu


def handle(N):
    return capi.Lattice(capi.make_params(N, phys(N)["dspa"], SQ_HALF, num_bin=4, num_bin_grav=4))


def field(N, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal((N, N, N)) + 1j * rng.standard_normal((N, N, N))


# 16 N^3 bytes against 16 MiB and chunks of 4 MiB: 96 below, 108 a remainder, 128 whole chunks, 162 more
# chunks than the ring has slots
@pytest.mark.parametrize("N", [96, 108, 128, 162])
def test_round_trip(N):
    print("[case] host copies", N, flush=True)
    f, g = field(N, 1), field(N, 2)
    for _ in range(2):  # the second handle makes the ring again
        with handle(N) as L:
            L.set_fields(f, g)
            a, b = L.get_fields()
            assert np.array_equal(a, f) and np.array_equal(b, g)
            rng = np.random.default_rng(3)
            A = rng.standard_normal((4, N, N, N // 2 + 1)) + 1j * rng.standard_normal((4, N, N, N // 2 + 1))
            L.set_gw_state(A)
            assert np.array_equal(L.gw_state(), A)


def test_odd_offset():
    print("[case] host copies, destination 8 bytes off", flush=True)
    N = 128
    f, g = field(N, 1), field(N, 2)
    with handle(N) as L:
        L.set_fields(f, g)
        out = np.zeros(2 * N ** 3 + 2)
        p = C.c_void_p(out.ctypes.data + 8)
        assert capi.lib().axg_get_fields(L._h, p, None, N ** 3) == 0
        assert np.array_equal(out[1:-1], f.ravel().view(np.float64)) and out[0] == 0 and out[-1] == 0


def test_two_threads():
    print("[case] host copies, two handles at once", flush=True)
    N, bad = 128, []

    def run(seed):
        f, g = field(N, seed), field(N, seed + 1)
        with handle(N) as L:
            for _ in range(4):
                L.set_fields(f, g)
                a, b = L.get_fields()
                if not (np.array_equal(a, f) and np.array_equal(b, g)):
                    bad.append(seed)

    t = [threading.Thread(target=run, args=(s,)) for s in (1, 11)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    assert not bad
