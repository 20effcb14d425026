"""String fits on a lattice with more strings than the eight-lane simplex kernel takes (one string per lane
there, in two kernels), and the eight-lane starts with counts that leave octets and waves part empty."""
import numpy as np
import pytest

import oracle as O
from axion_grav_amd import capi
from tests.conftest import SQ_HALF, phys

pytestmark = pytest.mark.gpu


def fit(prm, phi, pi, stream):
    with capi.Lattice(prm) as L:
        L.set_fields(phi, pi)
        f = L.get_fields()
        if stream:
            L.set_stream(*stream)
        cnt = L.defects()
        out = L.strings(21, 8)
        return f, int(cnt[0]), out, L.string_records()


def against_oracle(f, rec, count, dspa, stream):
    """The first `count` strings (the draws go by a string's index in site order) at the string tests' bar."""
    flags, _ = O.classify(f[0])
    idx = np.flatnonzero(flags & 1)
    only = np.zeros(flags.size, np.int8)
    only[idx[:count]] = 1
    kw = {"stream": stream} if stream else {}
    orec, _ = O.strings(f[0], f[1], only.reshape(flags.shape), 21, 8, dspa, **kw)
    assert len(orec) == min(count, len(idx))
    rel = np.abs(rec[: len(orec)] - orec) / np.maximum(1, np.abs(orec))
    assert rel.max() < 1e-5, rel.max()


@pytest.mark.parametrize("prec,stream", [(capi.FP32C, None), (capi.FP64, (7, 9, 12345))])
def test_one_string_per_lane(prec, stream, monkeypatch):
    print("[case] strings, lanes", prec, stream, flush=True)
    N = 192
    P = phys(N)
    prm = capi.make_params(N, P["dspa"], SQ_HALF, precision=prec, grav_spec=False)
    phi, _ = O.ic_flat(N, 3, 1.0, P["dwav"])
    pi = 0.3 * np.roll(phi, 7, 0)
    f, n, out, rec = fit(prm, phi, pi, stream)
    assert n > 16384
    for split in ("0", "1000"):
        monkeypatch.setenv("AXG_STRING_SPLIT", split)
        _, _, out2, rec2 = fit(prm, phi, pi, stream)
        assert np.array_equal(rec, rec2) and out["length"] == out2["length"]
    against_oracle(f, rec, 400, P["dspa"], stream)


# uncorrelated phases: string cells everywhere, 8^3 and 12^3 of them fit a few waves, the last one in part
@pytest.mark.parametrize("N,seed", [(8, 0), (8, 1), (12, 2), (16, 3)])
def test_few_strings(N, seed):
    print("[case] strings, few", N, seed, flush=True)
    P = phys(N)
    rng = np.random.default_rng(seed)
    phi, pi = (rng.standard_normal((N, N, N)) + 1j * rng.standard_normal((N, N, N)) for _ in range(2))
    f, n, _, rec = fit(capi.make_params(N, P["dspa"], SQ_HALF, grav_spec=False), phi, pi, None)
    assert n > 0 and len(rec) == n
    against_oracle(f, rec, n, P["dspa"], None)
