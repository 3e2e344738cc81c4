"""Volume -> sinogram gathers of volumes with long lines (needs an MI355X).

One line's slices past 2 GiB, and slices of 8 MiB a line: offsets that the
row-by-row gather does not hold, so such volumes go slice by slice.
"""
import numpy as np
import torch
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from pridediff_amd import load_radontorch
    return load_radontorch()


def test_lines_of_more_than_two_gib(rt):
    """32768 x 1 x 16500 voxels (a line: 2.16e9 bytes), zero but for the last 64
    slices, which the detector sees: the sinogram of those slices alone.  Both
    round every sum of about 50 pixels and 3 slices in FP32: relative L2 <= 1e-6."""
    w, dz, n, part, rows, cols = 32768, 2.0 ** -7, 16500, 64, 16, 700
    sid, sdd = 500.0, 1000.0
    pix = 2.0 ** -8
    z_top = n / 2 * dz
    ang = torch.tensor([0.0], device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(1)
    tail = torch.rand(1, 1, part, 1, w, device="cuda", generator=gen)

    def project(x, shift_z):
        opt = [w, 1, x.shape[2], cols, rows, pix, pix, dz, 0.2, dz * sdd / sid * 1.25, sid, sdd,
               0.0, 0.0, shift_z, 0.0, (z_top - part * dz / 2) * sdd / sid]
        return rt.ProjConeFlatDis3d(x, torch.tensor(opt), ang)

    want = project(tail, z_top - part * dz / 2).double()
    x = torch.zeros(1, 1, n, 1, w, device="cuda")
    x[:, :, -part:] = tail
    got = project(x, 0.0).double()
    err = float((got - want).norm() / want.norm())
    print(f"rel_l2 {err:.2e}", flush=True)
    assert float(want.abs().max()) > 0 and err <= 1e-6


@pytest.mark.parametrize("batch", [1, 2])
def test_slices_of_more_than_eight_mib_a_line(rt, batch):
    """2.2 million pixels on a line: relative L2 against 64 bits <= 5e-6 (sums
    of 2500 pixels in FP32)."""
    w, n, rows, cols = 2_200_000 // batch, 2, 5, 40
    g = O.Geom3D(w, 1, n, cols, rows, 1e-4, 1e-4, 1.0, 0.5, 1.0, 500.0, 1000.0)
    ang = np.array([0.0], dtype=np.float32)
    x = np.random.default_rng(2).random((batch, n, 1, w), dtype=np.float32)
    got = rt.ProjConeFlatDis3d(torch.from_numpy(x)[:, None].cuda(), torch.tensor(g.options()),
                               torch.from_numpy(ang).cuda())[:, 0].cpu().numpy()
    err = O.rel_l2(got, O.op3d("cone_flat", "proj", x, ang, g))
    print(f"batch {batch}: rel_l2 {err:.2e}", flush=True)
    assert err <= 5e-6
