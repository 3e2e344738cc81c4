"""Gather of fine bins, 2 x 2 pixels a thread (needs an MI355X).

Images large enough for it (from 1024 workgroups of 32 x 32 pixels on), odd
sizes in both directions, one and several chunks of views, a detector narrower
than the image, bins that are not finite: bit for bit the gather of one pixel a
thread, which a workgroup width chooses.
"""
import numpy as np
import pytest
import torch

from tests.test_gpu_routes_time import best_us

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from pridediff_amd import load_radontorch
    return load_radontorch()


def _plan(rt, scan, w, h, d, fine, views, batch, width):
    pix = 358.4 / max(w, h)
    det = pix / fine * (1.0 if scan == "para" else 1085.6 / 595.0) / (1085.6 if scan == "arc" else 1.0)
    opt = torch.tensor([w, h, d, pix, pix, det, 595.0, 1085.6, 0.3, -0.2, 0.1 * det])
    ang = torch.arange(views, device="cuda", dtype=torch.float32) * (2 * np.pi / views) + 0.11
    return rt.Plan2d(rt.SCAN[scan], opt, ang, batch, 0, -1, 0, 0, width)


@pytest.mark.parametrize("scan", ["para", "flat", "arc"])
@pytest.mark.parametrize("w,h,d,fine,views,batch", [
    (1025, 1023, 4500, 4.0, 7, 1), (1001, 1063, 2600, 4.2, 20, 2), (2111, 512, 6000, 6.0, 17, 1)])
def test_quads_equal_single_pixels(rt, scan, w, h, d, fine, views, batch):
    quads, pixels = (_plan(rt, scan, w, h, d, fine, views, batch, k) for k in (0, 16))
    gen = torch.Generator(device="cuda").manual_seed(w)
    y = torch.rand(batch, 1, views, d, device="cuda", generator=gen) - 0.3
    y[0, 0, 2, d // 2] = float("inf")
    y[0, 0, 3, d // 3] = float("nan")
    for op in [rt.PROJ_T, rt.BPROJ] + ([] if scan == "para" else [rt.BPROJ_W]):
        a, b = quads.run(op, y), pixels.run(op, y)
        assert torch.equal(torch.nan_to_num(a, nan=-1e30), torch.nan_to_num(b, nan=-1e30))


def test_large_images_take_quads(rt):
    """3000 x 3000 x 90 views, two bins a pixel: 0.8 of the time per pixel."""
    y = torch.rand(1, 1, 90, 6480, device="cuda")
    t = []
    for width in (0, 16):
        p = _plan(rt, "arc", 3000, 3000, 6480, 2.0, 90, 1, width)
        t.append(best_us(lambda: p.run(rt.PROJ_T, y), passes=3))
    print(f"quads {t[0]:.0f} us, per pixel {t[1]:.0f} us", flush=True)
    assert t[0] <= 0.92 * t[1]
