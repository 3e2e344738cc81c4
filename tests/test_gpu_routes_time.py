"""Calls beside the usual sizes take the kernel that suits them (needs an
MI355X): their time relative to a neighbouring call, best of several passes.
Each bound lies well between what the right and the wrong kernel measure, both
given with it."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from pridediff_amd import load_radontorch
    return load_radontorch()


def best_us(fn, passes=10, reps=5):
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    for _ in range(3):
        fn()
    times = []
    for _ in range(reps):
        a.record()
        for _ in range(passes):
            fn()
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b) / passes * 1e3)
    return min(times)


def forward3d(rt, n, cols, rows, columns_per_pixel, views, batch):
    pix = 256.0 / n
    opt = torch.tensor([n, n, n // 2, cols, rows, pix, pix, pix, pix * 1.5 / columns_per_pixel,
                        pix * 1.5, 1000.0, 1500.0, 0.2, -0.3, 0.1, 0.0, 0.3])
    ang = torch.arange(views, device="cuda", dtype=torch.float32) * (2 * np.pi / views) + 0.05
    x = torch.rand(batch, 1, n // 2, n, n, device="cuda")
    return best_us(lambda: rt.ProjConeFlatDis3d(x, opt, ang))


@pytest.mark.parametrize("batch", [1, 4])
def test_forward_of_one_detector_row(rt, batch):
    """One row against eight of a 128 x 128 x 64 volume, 120 views: 0.99 of
    the time where a chunk of eight rows is walked for it, 0.4 to 0.65 slice by
    slice."""
    one, eight = (forward3d(rt, 128, 180, r, 1.0, 120, batch) for r in (1, 8))
    print(f"batch {batch}: one row {one:.0f} us, eight {eight:.0f} us", flush=True)
    assert one <= 0.8 * eight


def test_forward_of_coarse_columns(rt):
    """Columns of two pixels against columns of one, four volumes of 128 x 128
    x 64, 90 views: 3.7 times the time row by row, 1.7 slice by slice."""
    coarse, fine = forward3d(rt, 128, 95, 80, 0.5, 90, 4), forward3d(rt, 128, 190, 80, 1.0, 90, 4)
    print(f"two pixels {coarse:.0f} us, one {fine:.0f} us", flush=True)
    assert coarse <= 2.5 * fine


def adjoint2d(rt, n, views, batch):
    pix = 358.4 / n
    opt = torch.tensor([n, n, int(1.44 * n), pix, pix, pix / 595.0, 595.0, 1085.6, 0.3, -0.2, 0.0])
    ang = torch.arange(views, device="cuda", dtype=torch.float32) * (2 * np.pi / views) + 0.11
    y = torch.rand(batch, 1, views, int(1.44 * n), device="cuda")
    return best_us(lambda: rt.ProjTransFanArcDis2d(y, opt, ang))


@pytest.mark.parametrize("n,views,batch,most", [(1024, 1, 1, 0.22), (512, 4, 16, 0.28)])
def test_adjoint_of_few_views(rt, n, views, batch, most):
    """Against 64 views: one view of 1024 x 1024 a third of the time where one
    workgroup forms the view's range table, an eighth without; 4 views of 16
    slices of 512 x 512 0.36 by the staged walk, 0.19 per pixel."""
    few, many = adjoint2d(rt, n, views, batch), adjoint2d(rt, n, 64, batch)
    print(f"{n} x {n} x {batch}: {views} views {few:.1f} us, 64 views {many:.1f} us", flush=True)
    assert few <= most * many


def test_adjoint_of_fine_fan_angles(rt):
    """4096 x 4096, 90 views, one bin a pixel, 8e-5 rad: as long as with a flat
    detector of that pitch, 1.8 of it where the guess of a pixel's first bin
    misses its window."""
    n, views, d = 4096, 90, 5888
    pix = 358.4 / n
    det = pix * 1085.6 / 595.0
    ang = torch.arange(views, device="cuda", dtype=torch.float32) * (2 * np.pi / views) + 0.11
    y = torch.rand(1, 1, views, d, device="cuda")
    t = {}
    for scan, fn, pitch in (("arc", rt.ProjTransFanArcDis2d, det / 1085.6),
                            ("flat", rt.ProjTransFanFlatDis2d, det)):
        opt = torch.tensor([n, n, d, pix, pix, pitch, 595.0, 1085.6, 0.3, -0.2, 0.0])
        t[scan] = best_us(lambda: fn(y, opt, ang), passes=2, reps=3)
    print(f"arc {t['arc']:.0f} us, flat {t['flat']:.0f} us", flush=True)
    assert t["arc"] <= 1.35 * t["flat"]


def test_adjoint3d_of_blocks_beyond_the_buffer(rt):
    """33 x 33 x 120 near the source, 60 views: most views' blocks of rows are
    too large for the LDS buffer at four instances.  Four volumes against one:
    3.3 times the time where those views run on 135 workgroups, 1.5 where they
    are split like the others."""
    w, dz, views, cols, sid, sdd, per = 33, 120, 60, 60, 120.0, 210.0, 2.3
    rows = int(dz * per * 1.3)
    opt = torch.tensor([w, w, dz, cols, rows, 1.0, 1.0, 1.0, 1.5 * sdd / sid * w / cols,
                        sdd / sid / per, sid, sdd, 0.0, 0.0, 0.0, 0.0, 0.0])
    ang = torch.arange(views, device="cuda", dtype=torch.float32) * (2 * np.pi / views) + 0.05
    t = []
    for batch in (4, 1):
        y = torch.rand(batch, 1, views, rows, cols, device="cuda")
        t.append(best_us(lambda: rt.ProjTransConeFlatDis3d(y, opt, ang)))
    print(f"four {t[0]:.0f} us, one {t[1]:.0f} us", flush=True)
    assert t[0] <= 2.3 * t[1]


def test_setup_of_uneven_batches(rt):
    """Plans of one instance, 16 views: 2048 x 2048 against 256 x 256, 4 times
    the time where one workgroup forms a view's ranges, 1.3 where several do."""
    import time
    ang = torch.arange(16, device="cuda", dtype=torch.float32) * 0.3
    t = {}
    for n in (2048, 256):
        opt = torch.tensor([n, n, int(1.44 * n), 358.4 / n, 358.4 / n, 358.4 / n / 595.0, 595.0,
                            1085.6, 0.0, 0.0, 0.0])
        t[n] = 1e9
        for _ in range(12):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            plan = rt.PlanBatch2d(rt.SCAN["arc"], [opt], [ang], 0)
            torch.cuda.synchronize()
            t[n] = min(t[n], (time.perf_counter() - t0) * 1e6)
            del plan
    print(f"2048: {t[2048]:.0f} us, 256: {t[256]:.0f} us", flush=True)
    assert t[2048] <= 2.5 * t[256]
