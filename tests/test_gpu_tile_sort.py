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


@pytest.mark.parametrize("per_tile,side,planes", [
    ([0, 1, 48, 49, 64, 300, 1280, 1281, 2560], 40, 1), ([2561, 4096, 5000, 8192, 9000, 16384], 16, 1),
    ([16385, 17000], 2, 1), ([20000, 24000], 4, 4)])
def test_a_frame_of_one_depth(per_tile, side, planes):
    """A plane facing the camera: the entries of every tile have the same depth
    bits, at the lengths of every instantiation and in many tiles, so that
    blocks share CUs; and lists past 16384 entries of four such planes, each
    plane a run of its own. The order is (depth, flatten id)."""
    lengths = np.resize(np.array(per_tile), side * side)
    rng = np.random.default_rng(lengths.size)
    tile = rng.permutation(np.repeat(np.arange(side * side), lengths))
    n = tile.size
    m = (np.stack([tile % side, tile // side], -1) * 16 + 8).astype(np.float32)[None]
    d = (2.0 ** rng.integers(0, planes, n)).astype(np.float32)
    out = gsplat().intersect_tile_offsets_forward(
        {"means2d": dev(m), "radii": dev(np.full((1, n, 2), 3, np.int32)), "depths": dev(d[None])}, 1, 16, side, side)
    order = np.lexsort((np.arange(n), d, tile))
    np.testing.assert_array_equal(host(out["flatten_ids"]), order.astype(np.int32))
    ids = (tile[order].astype(np.int64) << 32) | d[order].view(np.uint32)
    np.testing.assert_array_equal(host(out["isect_ids"]), ids)
    np.testing.assert_array_equal(host(out["tile_offsets"]).ravel(), np.cumsum(lengths) - lengths)


@pytest.mark.parametrize("images", [1, 2, 7, 32, 33, 1024, 1025])
def test_images_start_after_the_earlier_ones(images):
    """Offsets and lists over several images (a tile pass block per image up to
    1024 of them, one block for all beyond), one image empty, against a numpy
    enumeration."""
    rng = np.random.default_rng(images)
    n, tw, th = 300 if images < 100 else 7, 5, 3
    m = rng.uniform(-10, 90, (images, n, 2)).astype(np.float32)
    r = rng.integers(0, 30, (images, n, 2)).astype(np.int32)
    if images > 1:
        r[images // 2] = 0
    d = rng.uniform(0.2, 9.0, (images, n)).astype(np.float32)
    g = gsplat()
    out = g.intersect_tile_offsets_forward({"means2d": dev(m), "radii": dev(r), "depths": dev(d)}, images, 16, tw, th)
    rf = r.astype(np.float32)  # the operator's float32 sums: a float64 m - r can fall on the other side of a tile edge
    lo = np.clip(np.floor((m - rf) / 16), 0, [tw, th]).astype(int)
    hi = np.clip(np.ceil((m + rf) / 16), 0, [tw, th]).astype(int)
    rows = []
    for i in range(images):
        for k in range(n):
            if (r[i, k] > 0).all():
                rows += [(i * tw * th + y * tw + x, d[i, k].view(np.uint32), i * n + k)
                         for y in range(lo[i, k, 1], hi[i, k, 1]) for x in range(lo[i, k, 0], hi[i, k, 0])]
    rows = np.array(sorted(rows), np.int64).reshape(-1, 3)
    np.testing.assert_array_equal(host(out["flatten_ids"]), rows[:, 2])
    np.testing.assert_array_equal(host(out["tile_offsets"]).ravel(), np.searchsorted(rows[:, 0], np.arange(images * tw * th)))
    assert out["isect_ids"].numel() == len(rows)
