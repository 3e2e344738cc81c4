"""Routes beside the usual ones, each against 64 bits or against an independent
kernel (needs an MI355X).

* 3D adjoint by rows: views whose block of rows does not fit the LDS buffer are
  added by a second kernel, from global memory (tall volumes near the source).
* dd2d_run_noalloc where its scratch does not hold the staged walk's partial
  images, or its range table: one wavefront takes all chunks of views, or the
  op is gathered per pixel; the bits are dd2d_run's.
* The staged walk on irregular scans against the view-resolved kernel, which
  shares none of its staging.
* Workgroup widths of the per-pixel gather, where it runs.
* Uneven batches with the running-sum variant on instances of fine bins.
"""
import ctypes

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.test_zz_no_alloc import Geom, _run_both, lib  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from pridediff_amd import load_radontorch
    return load_radontorch()


# slices, rows per slice, batch: from a tenth to three quarters of the tiles and views of
# the cone-flat scan have too large a block (rows of an LDS block: 86 for one
# instance, 73 for two, 36 for four)
@pytest.mark.parametrize("dz,per_slice,batch", [(120, 2.3, 1), (200, 2.3, 1), (90, 2.3, 2),
                                                (160, 2.3, 2), (40, 2.3, 4), (90, 2.3, 3),
                                                (60, 1.5, 4)])
@pytest.mark.parametrize("scan", ["cone_flat", "cone_arc"])
def test_blocks_of_rows_beyond_the_buffer(rt, scan, dz, per_slice, batch):
    """Relative L2 <= 5e-6: a slice edge's row is rounded to FP32 at a few tens
    of rows, 2^-20 of a row of its neighbour's value."""
    w, h, views, cols, sid, sdd = 33, 30, 20, 60, 120.0, 210.0
    rows, pitch = int(dz * per_slice * 1.3), 1.5 * sdd / sid * w / cols
    g = O.Geom3D(w, h, dz, cols, rows, 1.0, 1.0, 1.0, pitch if scan == "cone_flat" else pitch / sdd,
                 sdd / sid / per_slice, sid, sdd)
    ang = (np.arange(views) * (2 * np.pi / views) + 0.05).astype(np.float32)
    y = np.random.default_rng(dz).random((batch, views, rows, cols), dtype=np.float32)
    name = {"cone_flat": "ConeFlatDis3d", "cone_arc": "ConeArcDis3d"}[scan]
    for op, fn in (("proj_t", "ProjTrans"), ("bproj_w", "BackProjWeighted")):
        got = getattr(rt, fn + name)(torch.from_numpy(y)[:, None].cuda(),
                                     torch.tensor(g.options(), dtype=torch.float32),
                                     torch.from_numpy(ang).cuda())[:, 0].cpu().numpy()
        err = O.rel_l2(got, O.op3d(scan, op, y, ang, g))
        print(f"{scan} {op} {dz} slices, batch {batch}: {err:.2e}", flush=True)
        assert err <= 5e-6


def _noalloc_geom(scan, n, d):
    pix = 358.4 / n
    det = pix * (1.0 if scan == 0 else 1085.6 / 595.0) / (1085.6 if scan == 2 else 1.0)
    return Geom(n, n, d, pix, pix, det, 595.0, 1085.6, 0.3, -0.2, 0.1 * det)


# size, bins, views, batch: 134 MB of partial images at most, 4 MB and more of
# them past the scratch; then a range table of 47 MB beside 32 MB of the rest
@pytest.mark.parametrize("n,d,views,batch", [(512, 736, 180, 8), (512, 736, 180, 16),
                                             (700, 1000, 100, 4), (2048, 2944, 360, 1)])
@pytest.mark.parametrize("scan", [0, 1, 2])
def test_noalloc_without_room_for_the_walks_memory(lib, scan, n, d, views, batch):  # noqa: F811
    g = _noalloc_geom(scan, n, d)
    for op in [1, 2] + ([] if scan == 0 else [4]):
        print(f"scan {scan} op {op} {n}x{n}, {views} views, batch {batch}", flush=True)
        a, b, ws_bytes = _run_both(lib, scan, op, g, batch, views, seed=op + n)
        assert ws_bytes > 64 << 20
        assert not torch.isnan(a).any()
        assert torch.equal(a, b)


@pytest.mark.parametrize("scan,geom", [("para", "ParaDis2d"), ("flat", "FanFlatDis2d"),
                                       ("arc", "FanArcDis2d")])
@pytest.mark.parametrize("w,h,d,batch", [(96, 61, 131, 1), (45, 130, 150, 4), (80, 80, 60, 9),
                                         (33, 47, 70, 16)])
def test_irregular_scans_equal_the_sum_over_views(rt, scan, geom, w, h, d, batch):
    """Shuffled, repeated and uneven angles, rectangles, shifted detectors: the
    walk against the view-resolved op added up in 64 bits.  Both round each of
    at most 61 views' terms and the walk its sums: relative L2 <= 1e-6; and
    against the oracle."""
    rng = np.random.default_rng(w + h)
    ang = np.concatenate([rng.uniform(-7, 7, 40), np.full(3, 1.25), np.linspace(0, 0.3, 18)])
    ang = rng.permutation(ang).astype(np.float32)
    pix = 358.4 / max(w, h)
    det = pix * (1.0 if scan == "para" else 1085.6 / 595.0) / (1085.6 if scan == "arc" else 1.0)
    g = O.Geom2D(w, h, d, pix, 0.9 * pix, det, 595.0, 1085.6, 7.3, -4.2, 3.3 * det)
    opt, a = torch.tensor(g.options()), torch.from_numpy(ang).cuda()
    y = rng.random((batch, 61, d), dtype=np.float32)
    yt = torch.from_numpy(y)[:, None].cuda()
    for name, op, what in ([("ProjTrans", rt.PROJ_T, "proj_t"), ("BackProj", rt.BPROJ, "bproj")] +
                           ([] if scan == "para" else [("BackProjWeighted", rt.BPROJ_W, "bproj_w")])):
        got = getattr(rt, name + geom)(yt, opt, a)[:, 0]
        views = rt.views2d(rt.SCAN[scan], op, yt, opt, a)
        want = views.reshape(batch, 61, h, w).double().sum(1)
        err = float((got.double() - want).norm() / want.norm())
        ref = O.rel_l2(got.cpu().numpy(), O.op2d(scan, what, y, ang, g, "f64"))
        print(f"{scan} {what} {w}x{h} batch {batch}: views {err:.2e}, oracle {ref:.2e}", flush=True)
        assert err <= 1e-6 and ref <= 1e-6


@pytest.mark.parametrize("tile", [1, 4, 16])
@pytest.mark.parametrize("fine,views", [(4.0, 40), (1.0, 9)])
def test_widths_of_the_per_pixel_gather(rt, tile, fine, views):
    """Bins too fine to stage, and few views: every width gives the same bits,
    and they are the oracle's to 1e-6 (sums of at most 40 views)."""
    w, h, batch = 70, 53, 16
    pix = 5.0
    det = pix / fine / 595.0
    d = int(80 * fine)
    g = O.Geom2D(w, h, d, pix, pix, det, 595.0, 1085.6, 0.3, -0.2, 0.1 * det)
    ang = (np.arange(views) * (2 * np.pi / views) + 0.11).astype(np.float32)
    y = np.random.default_rng(views).random((batch, views, d), dtype=np.float32)
    yt = torch.from_numpy(y)[:, None].cuda()
    outs = []
    for width in (0, 16, 32, 64):
        p = rt.Plan2d(rt.SCAN["arc"], torch.tensor(g.options()), torch.from_numpy(ang).cuda(),
                      batch, tile, -1, 0, 0, width)
        assert p.pixel_gather(rt.PROJ_T)
        outs.append(p.run(rt.PROJ_T, yt))
    assert all(torch.equal(o, outs[0]) for o in outs[1:])
    err = O.rel_l2(outs[0][:2, 0].cpu().numpy(), O.op2d("arc", "proj_t", y[:2], ang, g, "f64"))
    print(f"tile {tile}, {fine} bins a pixel, {views} views: {err:.2e}", flush=True)
    assert err <= 1e-6


@pytest.mark.parametrize("scan", ["para", "flat", "arc"])
def test_uneven_running_sums_of_fine_bins(scan):
    """ADJ_BLOCK_PREFIX on instances whose bins are too fine to stage (and one
    that is staged): running sums against 64 bits, relative L2 <= 2e-6 (knots
    in FP64; positions and sums of a 4-pixel run in FP32, once a view)."""
    from pridediff_amd import load_radontorch
    from pridediff_amd.batched import UnevenBatch2d
    from pridediff_amd.deeprecon.torch.projector import projector2d
    rt = load_radontorch()
    projs, angs, ys = [], [], []
    rng = np.random.default_rng(8)
    for i, (n, d, det) in enumerate(((70, 700, 0.5), (130, 900, 0.5), (41, 300, 0.4), (64, 150, 3.0))):
        projs.append(projector2d(n, d, 1.4, det, 595.0, 1085.6, scan_type=scan).cuda())
        v = 31 + 9 * i
        angs.append((np.arange(v) * (2 * np.pi / v) + 0.03).astype(np.float32))
        ys.append(rng.random((v, d), dtype=np.float32))
    ub = UnevenBatch2d(projs, [torch.from_numpy(a).cuda() for a in angs])
    ub.plan.set_variant(rt.ADJ_BLOCK_PREFIX)
    flat = ub.pack_sinos([torch.from_numpy(y).cuda() for y in ys])
    for op, what in (("projection_t", "proj_t"), ("backprojection", "bproj")):
        with torch.no_grad():
            outs = ub.unpack_images(getattr(ub, op)(flat))
        for P, a, y, o in zip(projs, angs, ys, outs):
            v = [float(t) for t in P.host_options().tolist()]
            g = O.Geom2D(int(v[0]), int(v[1]), int(v[2]), *v[3:])
            err = O.rel_l2(o.cpu().numpy()[None], O.op2d(scan, what, y[None], a, g, "f64"))
            print(f"{scan} {what} {g.W}: {err:.2e}", flush=True)
            assert err <= 2e-6
