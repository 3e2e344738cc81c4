"""3D gathers by detector rows where rows and slices have any size relative to
each other (needs an MI355X).

A helical view brings its own source radius, which the choice of a kernel does
not see: rows can be millions of slices high, and the other way round.  Every
loop over the slices of a row (the rows of a slice) ends at the volume's (the
detector's) own count.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from pridediff_amd import load_radontorch
    return load_radontorch()


@pytest.mark.parametrize("batch", [1, 2, 4])
def test_rows_of_millions_of_slices(rt, batch):
    """Detector a millionth of a millimetre from the source: the first row
    takes the upper half of the volume (2.2e7 slices from its middle on), the
    others nothing.  Sums of 8 slices of 16 pixels in FP32: relative L2 <= 5e-6."""
    sid, sdd, step = 100.0, 16.0 - 2.0 ** -10, 2.0 ** -20  # step: one ulp below 16
    g = O.Geom3D(16, 16, 16, 4, 8, 1.0, 1.0, 1.0, 0.02 * step / sdd, 0.25, sid, sdd, 0.0, 0.0,
                 0.0, 0.0, 1.0)
    ang = np.array([0.0, 1.5, 2.9], dtype=np.float32)
    spos = np.zeros((4, 3), dtype=np.float32)
    spos[1] = step - sdd
    assert np.float32(step - sdd) + np.float64(np.float32(sdd)) == step
    x = np.random.default_rng(3).random((batch, 16, 16, 16), dtype=np.float32)
    got = rt.ProjSpiralDis3d(torch.from_numpy(x)[:, None].cuda(),
                             torch.tensor(g.options(spiral=True), dtype=torch.float32),
                             torch.from_numpy(ang).cuda(), torch.from_numpy(spos).cuda())
    got = got[:, 0].cpu().numpy()
    want = O.op3d("spiral", "proj", x, ang, g, spos)
    assert np.abs(want[:, :, 0]).max() > 0 and not np.abs(want[:, :, 1:]).any()
    err = O.rel_l2(got, want)
    print(f"batch {batch}: rel_l2 {err:.2e}", flush=True)
    assert err <= 5e-6


@pytest.mark.parametrize("batch", [1, 2, 4])
def test_slices_of_millions_of_rows(rt, batch):
    """A source on the volume's first line of pixels: a slice there is 1.9e7
    rows.  The running sums bound the same rows by clamped differences; the
    other lines agree with them to their rounding (5e-6), that line to the
    rounding of its pixels' overlap (an FP32 fraction near 1 times 1e-5 of a
    pixel: 1e-2)."""
    sid, sdd = 120.0, 210.0
    g = O.Geom3D(8, 8, 8, 12, 20, 1.0, 1.0, 1.0, 0.05, 0.65, sid, sdd)
    ang = np.array([0.0, 0.7, 2.0], dtype=np.float32)
    spos = np.zeros((4, 3), dtype=np.float32)
    spos[1, 0] = np.float32(-116.5 + 2.0 ** -17)  # source at y = 3.5 + 2^-17 in view 0
    y = np.random.default_rng(4).random((batch, 3, 20, 12), dtype=np.float32)
    args = [torch.from_numpy(y)[:, None].cuda(),
            torch.tensor(g.options(spiral=True), dtype=torch.float32),
            torch.from_numpy(ang).cuda(), torch.from_numpy(spos).cuda()]
    rows = rt.ProjTransSpiralDis3d(*args)[:, 0].cpu()
    rt.set_compensated3d(1)
    try:
        sums = rt.ProjTransSpiralDis3d(*args)[:, 0].cpu()
    finally:
        rt.set_compensated3d(2)
    assert torch.isfinite(rows).all()
    for what, at, tol in (("other lines", slice(1, 8), 5e-6), ("first line", slice(0, 1), 1e-2)):
        a, b = rows[:, :, at].double(), sums[:, :, at].double()
        err = float((a - b).norm() / b.norm())
        print(f"batch {batch}, {what}: rel_l2 {err:.2e}", flush=True)
        assert err <= tol
