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
