"""The spherical harmonics operator on rows of exactly the active bases (whole
float4s per row at degrees 1 and 3, odd row lengths at 2 and 4; degree 0 has
the general kernels only): the same bits as on the leading bases of longer
rows, which take the general kernels, for whole and partial blocks of 64 rows,
masks, and with and without direction gradients; and views whose rows are not
16-byte aligned."""
import numpy as np
import pytest

from _helpers import dev, gsplat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degree", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000])
@pytest.mark.parametrize("masked", [False, True])
def test_whole_rows_equal_leading_bases(degree, n, masked):
    import torch

    g = gsplat()
    rng = np.random.default_rng(degree * 10 + n)
    A = (degree + 1) ** 2
    dirs = rng.normal(size=(n, 3)).astype(np.float32)
    dirs[0] = 0.0
    coeffs = rng.normal(size=(n, A, 3)).astype(np.float32)
    longer = np.concatenate([coeffs, rng.normal(size=(n, 2, 3)).astype(np.float32)], 1)
    v = dev(rng.normal(size=(n, 3)).astype(np.float32))
    extra = {"masks": dev(rng.random(n) < 0.7)} if masked else {}
    a = {"dirs": dev(dirs), "coeffs": dev(coeffs), **extra}
    b = {"dirs": dev(dirs), "coeffs": dev(longer), **extra}
    storage = torch.empty(n * A * 3 + 1, device="cuda")
    shifted = storage[1:].view(n, A, 3)
    shifted.copy_(a["coeffs"])
    c = {"dirs": a["dirs"], "coeffs": shifted, **extra}
    want = g.spherical_harmonics_forward(degree, b)
    assert torch.equal(g.spherical_harmonics_forward(degree, a), want)
    assert torch.equal(g.spherical_harmonics_forward(degree, c), want)
    for with_dirs in (True, False):
        wb = g.spherical_harmonics_backward(degree, b, {"v_colors": v}, with_dirs)
        for x in (a, c):
            got = g.spherical_harmonics_backward(degree, x, {"v_colors": v}, with_dirs)
            assert torch.equal(got["v_coeffs"], wb["v_coeffs"][:, :A])
            if with_dirs:
                assert torch.equal(got["v_dirs"], wb["v_dirs"])
