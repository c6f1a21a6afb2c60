"""The sort of one tile's list in LDS: the distribution over the range of the
depth bits and the radix passes it falls back to, at the list lengths where the
instantiations change and for depths that spread evenly, crowd a bin, tie, or
straddle the sign. The order is (depth bits as unsigned, flatten id), computed
by numpy; ids and flatten ids are exact."""
import numpy as np
import pytest

from _helpers import dev, gsplat, host

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 63, 255, 1279, 1280, 1281, 2560, 2561, 4096, 4097, 8192, 8193, 16384, 16385]


def _depths(kind, n, rng):
    if kind == "even":
        return rng.uniform(0.2, 12.0, n)
    if kind == "equal":
        return np.full(n, 3.5)
    if kind == "outlier":  # one far depth stretches the range over a narrow cluster
        d = rng.uniform(5.0, 5.001, n)
        d[n // 2] = 1e9
        return d
    if kind == "runs":  # runs of equal depths of 1 to 60, around the crowding limit
        return np.repeat(rng.uniform(1.0, 9.0, n), rng.integers(1, 61, n))[:n][rng.permutation(n)]
    d = rng.normal(0.0, 1.0, n)  # "signed": negative bits sort last, and both zeros
    d[: n // 3] = np.where(rng.random(n // 3) < 0.5, 0.0, -0.0)
    return d


@pytest.mark.parametrize("kind", ["even", "equal", "outlier", "runs", "signed"])
@pytest.mark.parametrize("n", LENGTHS)
def test_one_tile(n, kind):
    rng = np.random.default_rng(n)
    d = _depths(kind, n, rng).astype(np.float32)
    g = gsplat()
    m = np.full((1, n, 2), 8.0, np.float32)
    r = np.full((1, n, 2), 3, np.int32)
    out = g.intersect_tile_offsets_forward({"means2d": dev(m), "radii": dev(r), "depths": dev(d[None])}, 1, 16, 1, 1)
    bits = d.view(np.uint32)
    order = np.lexsort((np.arange(n), bits))
    np.testing.assert_array_equal(host(out["flatten_ids"]), order.astype(np.int32))
    ids = host(out["isect_ids"]).astype(np.uint64)
    np.testing.assert_array_equal((ids & 0xFFFFFFFF).astype(np.uint32), bits[order])
    assert host(out["tile_offsets"]).ravel().tolist() == [0]
