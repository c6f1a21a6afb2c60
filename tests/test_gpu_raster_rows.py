"""The rasterizer kernels with records in lanes (tile sides 8, 16 and 24, one to
four channels, no absolute gradients, lists long enough) against the oracle,
where their groups of 16 records, their batches of 128 and 256 entries, their
record classes and the forward's pixel blocks meet: list lengths around 16, 128
and 256 (the shortest take the kernels with pixels in lanes), every tile side,
opacities over the 0.99 cap, ill-conditioned conics, opacities over 1,
non-finite and overflowing values, and grids on both sides of the forward's
block sizes, of the backward's batches and of the rules that choose the kernel.

Tolerance: images 1e-4 and exact last contributors as elsewhere; the gradients'
usual bar, 1e-3 of each element or of 1% of the tensor's largest (both sides
round every pixel's terms in float32; the sums run in another order).
"""
import numpy as np
import pytest

from _helpers import assert_close_rel, dev, gsplat, host
from test_gpu_raster import GRAD_RTOL, IMG_ATOL, _oracle_fwd, _raster_inputs, make_scene

pytestmark = pytest.mark.gpu


def _check(oracle, s, W, H, ts, rng, finite=True):
    g = gsplat()
    got = g.rasterize_to_pixels_3dgs_forward(_raster_inputs(s), W, H, ts)
    exp = _oracle_fwd(oracle, s, W, H, ts)
    np.testing.assert_array_equal(host(got["last_ids"]), exp["last_ids"])
    for k in ("render_colors", "render_alphas"):
        a, e = host(got[k]), exp[k]
        np.testing.assert_array_equal(np.isfinite(a), np.isfinite(e), err_msg=k)
        np.testing.assert_allclose(a[np.isfinite(e)], e[np.isfinite(e)], rtol=0, atol=IMG_ATOL, err_msg=k)
    v_rc = rng.normal(size=exp["render_colors"].shape).astype(np.float32)
    v_ra = rng.normal(size=exp["render_alphas"].shape).astype(np.float32)
    bwd = g.rasterize_to_pixels_3dgs_backward(
        _raster_inputs(s), {"render_alphas": got["render_alphas"], "last_ids": got["last_ids"]},
        {"v_render_colors": dev(v_rc), "v_render_alphas": dev(v_ra)}, W, H, ts)
    want = oracle.raster_backward(s["means2d"], s["conics"], s["colors"], s["opacities"], s["tile_offsets"],
                                  s["flatten_ids"], W, H, ts, exp["render_alphas"], exp["last_ids"], v_rc, v_ra,
                                  backgrounds=s["backgrounds"], masks=s.get("masks"))
    for k in ("v_means2d", "v_conics", "v_colors", "v_opacities"):
        a, e = host(bwd[k]), want[k]
        if not finite:
            np.testing.assert_array_equal(np.isfinite(a), np.isfinite(e), err_msg=k)
            a, e = np.where(np.isfinite(e), a, 0), np.where(np.isfinite(e), e, 0)
        assert_close_rel(a, e, GRAD_RTOL, k)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 127, 129, 255, 256, 257, 529])
def test_list_lengths(oracle, n):
    """One tile whose list holds about n faint records (every group and batch remainder)."""
    rng = np.random.default_rng(n)
    s = make_scene(oracle, rng, 1, n, 16, 16, 16, 3, opac=(0.006, 0.03), scale=(4.0, 9.0))
    _check(oracle, s, 16, 16, 16, rng)


@pytest.mark.parametrize("ts,C,W,H,masks", [(8, 3, 61, 45, False), (16, 1, 50, 33, True), (16, 2, 70, 40, False),
                                            (24, 4, 75, 50, False), (32, 3, 97, 64, True), (16, 4, 33, 47, False)])
def test_tile_sides_and_channels(oracle, ts, C, W, H, masks):
    rng = np.random.default_rng(ts + C)
    s = make_scene(oracle, rng, 2, 900, W, H, ts, C, opac=(0.05, 0.9), masks=masks)
    _check(oracle, s, W, H, ts, rng)


@pytest.mark.parametrize("opac", [(0.9, 0.99), (0.97, 1.0), (1.0, 1.7)])
def test_capped_and_general_opacities(oracle, opac):
    """Groups with records over the cap and over 1 beside plain ones."""
    rng = np.random.default_rng(7)
    s = make_scene(oracle, rng, 1, 600, 48, 48, 16, 3, opac=(0.05, 0.6), scale=(1.0, 3.0))
    pick = rng.random(s["opacities"].shape) < 0.2
    s["opacities"] = np.where(pick, rng.uniform(*opac, s["opacities"].shape), s["opacities"]).astype(np.float32)
    _check(oracle, s, 48, 48, 16, rng)


def test_ill_conditioned_and_non_finite_records(oracle):
    """Records of the general class in groups of plain ones: conics close to
    singular, not positive definite and huge, infinite and NaN means and colours."""
    rng = np.random.default_rng(11)
    W = H = 48
    s = make_scene(oracle, rng, 1, 500, W, H, 16, 3, opac=(0.05, 0.6), scale=(1.0, 4.0))
    con = s["conics"].reshape(-1, 3)
    con[3] = [0.2, 0.199999, 0.2]
    con[40] = [0.2, 0.3, 0.2]
    con[77] = [3.0e7, 0.0, 2.0e7]
    con[120] = [1.0e-18, 0.0, 0.3]
    mean = s["means2d"].reshape(-1, 2)
    mean[200] = [np.inf, 20.0]
    s["colors"].reshape(-1, 3)[250, 1] = np.inf
    s["colors"].reshape(-1, 3)[300, 2] = np.nan
    _check(oracle, s, W, H, 16, rng, finite=False)


def test_forward_block_sizes_agree(oracle):
    """The same image rendered as one of 1, 30 and 80 copies (12, 360 and 960
    tiles: 4x4, 8x4 and 8x8 pixel blocks per wave) comes out bit for bit."""
    import torch

    rng = np.random.default_rng(3)
    W, H, ts, n = 60, 47, 16, 800
    s = make_scene(oracle, rng, 1, n, W, H, ts, 3, opac=(0.05, 0.999), scale=(1.0, 6.0))
    _check(oracle, s, W, H, ts, rng)
    g = gsplat()
    one = _raster_inputs(s)
    ref = g.rasterize_to_pixels_3dgs_forward(one, W, H, ts)
    m = one["flatten_ids"].numel()
    for copies in (30, 80):
        many = {k: v.repeat(copies, *([1] * (v.dim() - 1))) for k, v in one.items() if k != "flatten_ids"}
        step = torch.arange(copies, device="cuda", dtype=torch.int32)
        many["tile_offsets"] = many["tile_offsets"] + (step * m)[:, None, None]
        many["flatten_ids"] = (one["flatten_ids"][None] + (step * n)[:, None]).reshape(-1).contiguous()
        got = g.rasterize_to_pixels_3dgs_forward(many, W, H, ts)
        for k in ("render_colors", "render_alphas"):
            assert torch.equal(got[k], ref[k].expand_as(got[k])), (copies, k)
        want = torch.where(ref["render_alphas"][..., 0] > 0, ref["last_ids"] + (step * m)[:, None, None], 0)
        assert torch.equal(got["last_ids"], want.to(got["last_ids"].dtype)), copies


def _check_backward_stays_local(oracle, s, W, H, v_rc, v_ra):
    """The backward's non-finite gradients are the oracle's: a pixel's values
    reach only the Gaussians that it takes."""
    exp = _oracle_fwd(oracle, s, W, H, 16)
    bwd = gsplat().rasterize_to_pixels_3dgs_backward(
        _raster_inputs(s), {"render_alphas": dev(exp["render_alphas"]), "last_ids": dev(exp["last_ids"])},
        {"v_render_colors": dev(v_rc), "v_render_alphas": dev(v_ra)}, W, H, 16)
    want = oracle.raster_backward(s["means2d"], s["conics"], s["colors"], s["opacities"], s["tile_offsets"],
                                  s["flatten_ids"], W, H, 16, exp["render_alphas"], exp["last_ids"], v_rc, v_ra,
                                  backgrounds=s["backgrounds"])
    for k in ("v_means2d", "v_conics", "v_colors", "v_opacities"):
        a, e = host(bwd[k]), want[k]
        np.testing.assert_array_equal(np.isfinite(a), np.isfinite(e), err_msg=k)
        fin = np.isfinite(e)
        assert fin.mean() > 0.8, k
        assert_close_rel(np.where(fin, a, 0), np.where(fin, e, 0), GRAD_RTOL, k)
    return want


@pytest.mark.parametrize("opac", [(0.05, 0.9), (0.5, 1.0)])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_non_finite_alpha_cotangents_stay_local(oracle, value, opac):
    """NaN and inf in the alpha cotangents of single pixels whose colour
    cotangents are finite, in groups without and with records over the cap."""
    rng = np.random.default_rng(29)
    W = H = 96
    s = make_scene(oracle, rng, 1, 1200, W, H, 16, 3, opac=opac)
    v_rc = rng.normal(size=(1, H, W, 3)).astype(np.float32)
    v_ra = rng.normal(size=(1, H, W, 1)).astype(np.float32)
    v_ra[0, 40, 41] = value
    v_ra[0, 70, 12] = -value
    want = _check_backward_stays_local(oracle, s, W, H, v_rc, v_ra)
    assert not np.isfinite(want["v_opacities"]).all()


def test_far_finite_means_give_no_gradient(oracle):
    """Finite means so far away that the square of their distance overflows:
    never culled, taken by no pixel, and without a gradient."""
    rng = np.random.default_rng(31)
    W = H = 48
    s = make_scene(oracle, rng, 1, 500, W, H, 16, 3, opac=(0.05, 0.6), scale=(1.0, 4.0))
    mean = s["means2d"].reshape(-1, 2)
    mean[100] = [1.0e31, 20.0]
    mean[222] = [20.0, -3.0e37]
    mean[333] = [-2.0e20, 5.0e19]
    s["conics"].reshape(-1, 3)[333] = [0.2, 0.199999, 0.2]
    v_rc = rng.normal(size=(1, H, W, 3)).astype(np.float32)
    v_ra = rng.normal(size=(1, H, W, 1)).astype(np.float32)
    want = _check_backward_stays_local(oracle, s, W, H, v_rc, v_ra)
    assert all(np.isfinite(want[k]).all() for k in ("v_means2d", "v_conics", "v_colors", "v_opacities"))
    assert (want["v_conics"].reshape(-1, 3)[[100, 222, 333]] == 0).all()


@pytest.mark.parametrize("color,cotangent,background", [(1.0e30, 1.0e20, 0.1), (0.5, 1.0e20, 1.0e30), (1.0e34, 1.0e12, 0.1)])
def test_overflowing_products_stay_local(oracle, color, cotangent, background):
    """Finite colours, backgrounds and cotangents whose products overflow at two
    pixels, there beyond 1e43, so that every order of the products with T > 1e-4
    overflows, and stay below 1e36 at the others."""
    rng = np.random.default_rng(37)
    W = H = 96
    s = make_scene(oracle, rng, 1, 1200, W, H, 16, 3)
    s["colors"][0, [5, 700]] = color
    s["backgrounds"][:] = background
    v_rc = rng.normal(size=(1, H, W, 3)).astype(np.float32)
    v_rc[0, 40, 41] = cotangent
    v_rc[0, 70, 12] = -cotangent
    v_ra = rng.normal(size=(1, H, W, 1)).astype(np.float32)
    _check_backward_stays_local(oracle, s, W, H, v_rc, v_ra)


def _pad_lists(s, pad):
    """The scene with `pad` entries of an added Gaussian of opacity 0 at the end of
    every tile's list: the same image and gradients, longer lists."""
    n = s["opacities"].shape[1]
    offs = s["tile_offsets"].reshape(-1).astype(np.int64)
    ends = np.append(offs[1:], s["flatten_ids"].size)
    at = np.repeat(ends, pad)
    out = dict(s)
    out["flatten_ids"] = np.insert(s["flatten_ids"], at, n).astype(np.int32)
    out["tile_offsets"] = (offs + np.arange(offs.size) * pad).astype(np.int32).reshape(s["tile_offsets"].shape)
    for k in ("means2d", "conics", "colors", "opacities"):
        last = np.ones_like(s[k][:, :1]) * (0.0 if k == "opacities" else 1.0)
        out[k] = np.concatenate([s[k], last.astype(np.float32)], 1)
    return out


@pytest.mark.parametrize("ts,C,W,H,pads", [
    (16, 3, 64, 48, [40]), (16, 4, 256, 240, [40]), (16, 3, 448, 400, [60]), (16, 4, 512, 496, [140]),
    (16, 1, 512, 496, [40]), (16, 3, 720, 560, [100, 300]), (16, 4, 720, 560, [100]), (8, 2, 200, 160, [40]),
    (8, 3, 400, 400, [40]), (8, 3, 600, 520, [140]), (24, 3, 120, 96, [40]), (24, 4, 700, 720, [40]),
    (24, 2, 700, 720, [300])])
def test_kernels_for_short_and_long_lists_agree(oracle, ts, C, W, H, pads):
    """Both sides of the lines by entries per tile, on grids of each of the rules'
    sizes: short lists, and the same lists lengthened past the line by entries
    that no pixel takes. The images are the same bits; the gradients differ by
    the order of their sums."""
    import torch

    rng = np.random.default_rng(W + C)
    tiles = -(-W // ts) * -(-H // ts)
    n = max(tiles if ts == 8 else 2 * tiles, 60)
    s = make_scene(oracle, rng, 1, n, W, H, ts, C, opac=(0.05, 0.999), scale=(0.5, 2.5))
    v_rc = dev(rng.normal(size=(1, H, W, C)).astype(np.float32))
    v_ra = dev(rng.normal(size=(1, H, W, 1)).astype(np.float32))
    g = gsplat()
    fwd, bwd = [], []
    for x in [s] + [_pad_lists(s, pad) for pad in pads]:
        inp = _raster_inputs(x)
        f = g.rasterize_to_pixels_3dgs_forward(inp, W, H, ts)
        bwd.append(g.rasterize_to_pixels_3dgs_backward(
            inp, {"render_alphas": f["render_alphas"], "last_ids": f["last_ids"]},
            {"v_render_colors": v_rc, "v_render_alphas": v_ra}, W, H, ts))
        first = inp["tile_offsets"].repeat_interleave(ts, 1).repeat_interleave(ts, 2)[:, :H, :W]
        f["last_ids"] = torch.where(f["last_ids"] > 0, f["last_ids"] - first, 0)
        fwd.append(f)
    for f, b in zip(fwd[1:], bwd[1:]):
        for k in ("render_colors", "render_alphas"):
            assert torch.equal(f[k], fwd[0][k]), k
        taken = fwd[0]["render_alphas"][..., 0] > 0
        assert torch.equal(f["last_ids"][taken], fwd[0]["last_ids"][taken])
        for k in ("v_means2d", "v_conics", "v_colors", "v_opacities"):
            assert (b[k][:, n] == 0).all(), k
            assert_close_rel(host(b[k][:, :n]), host(bwd[0][k]), GRAD_RTOL, k)


@pytest.mark.parametrize("C", [3, 4])
@pytest.mark.parametrize("n", [129, 200, 255, 257, 529])
def test_batches_of_many_tiles(oracle, n, C):
    """1100 copies of one tile's image: batches of 128 entries (lists below 256 on
    such a grid, and four channels) and of 256, with records that touch some of a tile's
    waves only, so that part-filled groups carry over. Every copy's gradients
    are the single image's, which the oracle's confirm."""
    import torch

    rng = np.random.default_rng(n + C)
    s = make_scene(oracle, rng, 1, n, 16, 16, 16, C, opac=(0.006, 0.05), scale=(0.6, 2.0))
    s["means2d"] = rng.uniform(0, 16, s["means2d"].shape).astype(np.float32)
    s["flatten_ids"] = rng.permutation(n).astype(np.int32)
    s["tile_offsets"] = np.zeros_like(s["tile_offsets"])
    _check(oracle, s, 16, 16, 16, rng)
    g = gsplat()
    one = _raster_inputs(s)
    copies = 1100
    many = {k: v.repeat(copies, *([1] * (v.dim() - 1))) for k, v in one.items() if k != "flatten_ids"}
    step = torch.arange(copies, device="cuda", dtype=torch.int32)
    many["tile_offsets"] = many["tile_offsets"] + (step * n)[:, None, None]
    many["flatten_ids"] = (one["flatten_ids"][None] + (step * n)[:, None]).reshape(-1).contiguous()
    cot = [dev(rng.normal(size=(1, 16, 16, c)).astype(np.float32)) for c in (C, 1)]
    out = []
    for inp, k in ((one, 1), (many, copies)):
        f = g.rasterize_to_pixels_3dgs_forward(inp, 16, 16, 16)
        out.append(g.rasterize_to_pixels_3dgs_backward(
            inp, {"render_alphas": f["render_alphas"], "last_ids": f["last_ids"]},
            {"v_render_colors": cot[0].repeat(k, 1, 1, 1), "v_render_alphas": cot[1].repeat(k, 1, 1, 1)}, 16, 16, 16))
    for k in ("v_means2d", "v_conics", "v_colors", "v_opacities"):
        # one tile per image: each sum is rounded once per batch, whatever the batches
        a, b = host(out[1][k]), host(out[0][k])
        assert_close_rel(a, np.broadcast_to(b, a.shape), 1e-5, k)
