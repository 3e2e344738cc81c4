"""Staged walk of the 2D sinogram -> image ops (needs an MI355X).

Sizes where it can go wrong: one pixel tile and remainders of it, few and
many views (one chunk, uneven chunks), bins from a third of a pixel (tiles of
fewer rows, then the per-pixel gather) to four pixels, detectors narrower
than the image, every instance tile; and values that are not finite.

Tolerance: every product rounds a weight (difference of two fractions in
[0, 1], half an ulp each, times the pixel weight) and itself, about
3 * 2^-24 relative, and a pixel's sum of up to 8 chunks of n views rounds
sqrt(n) ulps of its running value; at 200 views that stays under
10 * 2^-24 = 6e-7 of the result's norm, so relative L2 <= 1e-6.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

NAMES = {"proj_t": "ProjTrans", "bproj": "BackProj", "bproj_w": "BackProjWeighted"}
GEOMS = {"para": "ParaDis2d", "flat": "FanFlatDis2d", "arc": "FanArcDis2d"}


def _geom(scan, w, h, d, fine):
    """`fine`: bins per pixel at the isocentre."""
    pix = 358.4 / max(w, h)
    mag = 1.0 if scan == "para" else 1085.6 / 595.0
    det = pix / fine * mag / (1085.6 if scan == "arc" else 1.0)
    return O.Geom2D(w, h, d, pix, pix, det, 595.0, 1085.6, 0.3, -0.2, 0.1 * det)


def _op(scan, op, y, ang, g):
    from pridediff_amd import load_radontorch
    fn = getattr(load_radontorch(), NAMES[op] + GEOMS[scan])
    out = fn(torch.from_numpy(y)[:, None].cuda(), torch.tensor(g.options()),
             torch.from_numpy(ang).cuda())
    return out[:, 0]


CASES = [  # width, height, bins, bins per pixel, views, batch
    (16, 16, 24, 1.0, 7, 1), (17, 9, 25, 1.0, 16, 2), (1, 40, 60, 1.0, 9, 1),
    (61, 33, 97, 1.1, 66, 3), (48, 50, 30, 0.3, 64, 5), (47, 64, 101, 1.6, 67, 16),
    (40, 40, 100, 2.0, 40, 4), (33, 47, 190, 2.8, 33, 9), (40, 24, 150, 4.0, 24, 2),
    (64, 64, 20, 0.5, 200, 1), (130, 70, 140, 1.2, 61, 7)]


@pytest.mark.parametrize("w,h,d,fine,views,batch", CASES)
@pytest.mark.parametrize("scan", ["para", "flat", "arc"])
def test_walk_matches_oracle(scan, w, h, d, fine, views, batch):
    g = _geom(scan, w, h, d, fine)
    rng = np.random.default_rng(w * 1000 + h)
    y = rng.random((batch, views, d), dtype=np.float32)
    ang = ((np.arange(views) * (2 * np.pi / views)) + 0.11).astype(np.float32)
    for op in ["proj_t", "bproj"] + ([] if scan == "para" else ["bproj_w"]):
        print(f"{scan} {op} {w}x{h}, {d} bins, {views} views, batch {batch}", flush=True)
        got = _op(scan, op, y, ang, g)
        want = O.op2d(scan, op, y, ang, g, "f64")
        err = O.rel_l2(got.cpu().numpy(), want)
        print(f"rel_l2 {err:.2e}", flush=True)
        assert err <= 1e-6
        # a slice alone gets the bits it gets in the batch
        assert torch.equal(_op(scan, op, y[-1:], ang, g)[0], got[-1])


@pytest.mark.parametrize("batch", [1, 4, 8, 16])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_walk_keeps_values_that_are_not_finite_local(bad, batch):
    """One such bin reaches exactly the pixels that it touches: every other
    pixel is as with a zero there, bit for bit."""
    g = _geom("arc", 50, 37, 70, 1.0)
    views, rng = 40, np.random.default_rng(5)
    ang = (np.arange(views) * (2 * np.pi / views) + 0.07).astype(np.float32)
    y = rng.random((batch, views, 70), dtype=np.float32) + 0.5
    one = np.zeros_like(y[:1])
    one[0, 13, 33] = 1.0
    hit = (O.op2d("arc", "proj_t", one, ang, g, "f64")[0] > 0)
    y[0, 13, 33] = 0.0
    clean = _op("arc", "proj_t", y, ang, g).cpu().numpy()
    y[0, 13, 33] = bad
    got = _op("arc", "proj_t", y, ang, g).cpu().numpy()
    assert hit.any() and not np.isfinite(got[0][hit]).any()
    assert np.array_equal(got[0][~hit], clean[0][~hit])
    assert np.array_equal(got[1:], clean[1:])
