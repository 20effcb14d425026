"""The wall fits' direction search where several directions are least: flat walls midway between sites leave the
plane's two normals exactly equal, walls along axes and diagonals put the grid's directions in symmetric
pairs; and random cells of every number of edge points."""
import numpy as np
import pytest

import oracle as O
from axion_grav_amd import capi
from tests.conftest import SQ_HALF, phys

pytestmark = pytest.mark.gpu


def planes(N):
    x = np.arange(N)
    z, y, x = np.meshgrid(x, x, x, indexing="ij")
    return {"x": x + 0 * y, "y": y + 0 * x, "z": z + 0 * x, "xy": x + y, "xyz": x + y + z, "xz": x - z}


# the bar of the walls' parity test (last-bit differences of sin, cos and atan2 against libm, which also decide
# which of several equal directions comes out: on the flat walls, whose equal directions are turns about
# z by a grid angle and reflections, the height of the direction, its goodness of fit and the area)
@pytest.mark.parametrize("kind", ["x", "y", "z", "xy", "xyz", "xz", "random"])
def test_walls_match_oracle(kind):
    print("[case] wall search", kind, flush=True)
    N = 16
    P = phys(N)
    rng = np.random.default_rng(7)
    if kind == "random":
        ph = rng.uniform(-0.45 * np.pi, 0.45 * np.pi, (N, N, N)) + np.pi * (rng.random((N, N, N)) < 0.5)
    else:
        # the phase crosses pi between the sites where the coordinate passes a multiple of N / 2
        c = (planes(N)[kind] + 0.5) * 2 * np.pi * 2 / N
        ph = np.pi + 0.9 * np.sin(c)
    phi = (1 + 0.2 * rng.random((N, N, N))) * np.exp(1j * ph)
    with capi.Lattice(capi.make_params(N, P["dspa"], SQ_HALF, grav_spec=False)) as L:
        L.set_fields(phi, phi)
        cells = L.defects()
        try:
            L.walls()
        except capi.AxgError:
            pass  # cells with fewer than three crossings: the reference's stop; the records are there
        rec = L.wall_records()
    flags, _ = O.classify(phi)
    orec, _ = O.walls(phi, flags)[:2]
    assert len(rec) == len(orec) == cells[1] > 0
    if kind != "random":
        rec, orec = np.abs(rec[:, 5:]), np.abs(orec[:, 5:])
    assert (np.abs(rec - orec) / np.maximum(1, np.abs(orec))).max() < 1e-9
