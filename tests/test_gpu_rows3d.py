"""3D gathers by detector rows, both directions (needs an MI355X).

Sizes where the gather can go wrong: volumes of one pixel tile and remainders
of it, slice chunks with remainders, from two fifths of a row to just under
three rows per slice (windows of 2, 3 and 4 rows), a source that comes nearer
than the geometry says (more rows than any window), detectors shorter and
narrower than the volume, few views (not split) and many (split over
workgroups), and a batch per instance tile.

Tolerance: a slice edge's row coordinate is rounded to FP32 at a few tens of
rows (2^-20 of a row); it moves that much of a row's value from one slice to
the next, so with values of order one a sum is off by about 2^-20 / d of its
size, at d = 0.4 rows per slice 2.4e-6; relative L2 <= 5e-6.  The forward
rounds a row edge's slice coordinate the same way.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

NAMES = {"cone_flat": "ConeFlatDis3d", "cone_arc": "ConeArcDis3d", "spiral": "SpiralDis3d"}
OPS = {"proj_t": "ProjTrans", "bproj": "BackProj", "bproj_w": "BackProjWeighted"}
TO_SINO = {"proj": "Proj", "bproj_t": "BackProjTrans", "bproj_tw": "BackProjTransWeighted"}


@pytest.fixture(scope="module")
def rt():
    from pridediff_amd import load_radontorch
    return load_radontorch()


def _op(rt, scan, op, y, ang, g, spos):
    opt = torch.tensor(g.options(spiral=scan == "spiral"), dtype=torch.float32)
    args = [torch.from_numpy(y)[:, None].cuda(), opt, torch.from_numpy(ang).cuda()]
    if scan == "spiral":
        args.append(torch.from_numpy(spos).cuda())
    return getattr(rt, {**OPS, **TO_SINO}[op] + NAMES[scan])(*args)[:, 0].cpu().numpy()


# width, height, slices, columns, rows, rows per slice, nearest radius shift, views, batch
CASES = [
    (16, 16, 16, 30, 30, 1.0, 0.0, 7, 1),
    (17, 5, 1, 34, 3, 0.4, 0.0, 24, 2),
    (37, 21, 19, 64, 24, 0.9, 0.0, 40, 3),
    (20, 33, 35, 50, 66, 1.5, 0.0, 30, 2),
    (33, 18, 9, 26, 11, 2.3, 0.0, 25, 4),
    (12, 40, 24, 60, 20, 2.3, 0.0, 64, 1),
    (24, 24, 11, 40, 40, 2.2, -45.0, 20, 2),
]


def _geom(scan, w, h, dz, cols, rows, per_slice, shift, views):
    sid, sdd = 120.0, 210.0
    pitch = 1.5 * sdd / sid * max(w, h) / cols
    row = sdd / sid / per_slice
    g = O.Geom3D(w, h, dz, cols, rows, 1.0, 1.1, 1.0,
                 pitch if scan == "cone_flat" else pitch / sdd, row, sid, sdd, 0.2, -0.3,
                 0.1 if scan != "spiral" else 0.0, 0.0, 0.3)
    ang = (np.arange(views) * (2 * np.pi / views) + 0.05).astype(np.float32)
    spos = None
    if scan == "spiral":
        spos = np.stack([np.linspace(-4, 4, views), np.full(views, shift),
                         0.01 * np.cos(np.arange(views)), 0.2 * np.ones(views)]).astype(np.float32)
    return g, ang, spos


@pytest.mark.parametrize("w,h,dz,cols,rows,per_slice,shift,views,batch", CASES)
@pytest.mark.parametrize("scan", ["cone_flat", "cone_arc", "spiral"])
def test_rows_match_oracle(rt, scan, w, h, dz, cols, rows, per_slice, shift, views, batch):
    g, ang, spos = _geom(scan, w, h, dz, cols, rows, per_slice, shift, views)
    rng = np.random.default_rng(w * 100 + dz)
    y = rng.random((batch, views, rows, cols), dtype=np.float32)
    for op in OPS:
        print(f"{scan} {op} {w}x{h}x{dz}, {cols}x{rows}, {views} views, batch {batch}", flush=True)
        want = O.op3d(scan, op, y, ang, g, spos)
        got = _op(rt, scan, op, y, ang, g, spos)
        err = O.rel_l2(got, want)
        print(f"rel_l2 {err:.2e}", flush=True)
        assert err <= 5e-6
        # from global memory: the same rows, weights and order
        rt.set_adjoint_staging3d(0)
        try:
            unstaged = _op(rt, scan, op, y, ang, g, spos)
        finally:
            rt.set_adjoint_staging3d(2)
        err = O.rel_l2(unstaged, want)
        print(f"from global memory {err:.2e}", flush=True)
        assert err <= 5e-6
        if views < 16:  # one part: no partial volumes
            assert np.array_equal(got, unstaged)


# more: two and more slices per row near the far corner, a source that moves
# away (more slices than the host sees), rows up to the slice-major path, and
# enough wavefronts for the 16-row form
FORWARD = CASES + [
    (20, 18, 30, 34, 9, 0.55, 0.0, 12, 2),
    (20, 18, 30, 34, 9, 0.62, 60.0, 12, 1),
    (18, 20, 26, 30, 5, 0.3, 0.0, 12, 4),
    (16, 18, 20, 130, 33, 1.4, 0.0, 700, 1),
    (16, 18, 20, 130, 33, 1.4, 0.0, 700, 2),
]


@pytest.mark.parametrize("w,h,dz,cols,rows,per_slice,shift,views,batch", FORWARD)
@pytest.mark.parametrize("scan", ["cone_flat", "cone_arc", "spiral"])
def test_forward_rows_match_oracle(rt, scan, w, h, dz, cols, rows, per_slice, shift, views, batch):
    g, ang, spos = _geom(scan, w, h, dz, cols, rows, per_slice, shift, views)
    rng = np.random.default_rng(w * 100 + dz + 1)
    x = rng.random((batch, dz, h, w), dtype=np.float32)
    for op in TO_SINO:
        print(f"{scan} {op} {w}x{h}x{dz}, {cols}x{rows}, {views} views, batch {batch}", flush=True)
        got = _op(rt, scan, op, x, ang, g, spos)
        err = O.rel_l2(got, O.op3d(scan, op, x, ang, g, spos))
        print(f"rel_l2 {err:.2e}", flush=True)
        assert err <= 5e-6
