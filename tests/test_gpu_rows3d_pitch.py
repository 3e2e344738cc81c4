"""3D gathers by detector rows where rows and slices have the same pitch
(needs an MI355X).

On the line through the isocentre a row is then one, two or three slices (or
a slice so many rows) to the last bit, and every edge lies within a rounding
of a cell boundary.  On either side of it, the gathers have to put a row's
weight on the slices that it meets.

Tolerance as for other pitches: an edge's coordinate is rounded to FP32 at a
few tens of cells (2^-20 of a cell), which moves that much of a value from one
cell to the next: relative L2 <= 5e-6.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

NAMES = {"cone_flat": "ConeFlatDis3d", "cone_arc": "ConeArcDis3d"}
SID, SDD, ROW = 1000.0, 1500.0, 1.2


@pytest.mark.parametrize("dz,n", [(0.8, 32), (0.8, 64), (1.6, 32), (2.4, 30), (0.4, 40)])
@pytest.mark.parametrize("batch", [1, 2, 4])
@pytest.mark.parametrize("scan", ["cone_flat", "cone_arc"])
def test_matched_pitch(scan, dz, n, batch):
    """dz = 0.8: one row per slice; 1.6, 2.4: two, three; 0.4: a row of two
    slices (the width of the three-slice window)."""
    from pridediff_amd import load_radontorch
    rt = load_radontorch()
    rows = max(1, round(n * dz / 0.8))
    g = O.Geom3D(65, 65, n, 96, rows, 0.8, 0.8, dz,
                 1.2 if scan == "cone_flat" else 1.2 / SDD, ROW, SID, SDD)
    ang = np.array([0.0, np.pi / 2, 0.3, np.pi, 4.0], dtype=np.float32)
    rng = np.random.default_rng(int(dz * 10) + n)
    opt = torch.tensor(g.options(), dtype=torch.float32)
    for op, fn, shape in (("proj", "Proj", (batch, n, 65, 65)),
                          ("proj_t", "ProjTrans", (batch, ang.size, rows, 96)),
                          ("bproj_w", "BackProjWeighted", (batch, ang.size, rows, 96))):
        x = rng.random(shape, dtype=np.float32)
        got = getattr(rt, fn + NAMES[scan])(torch.from_numpy(x)[:, None].cuda(), opt,
                                            torch.from_numpy(ang).cuda())[:, 0].cpu().numpy()
        err = O.rel_l2(got, O.op3d(scan, op, x, ang, g))
        print(f"{scan} {op} dz {dz} x {n}, {rows} rows, batch {batch}: rel_l2 {err:.2e}", flush=True)
        assert err <= 5e-6
