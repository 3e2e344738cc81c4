"""2D sinogram -> image ops with few views (needs an MI355X).

A call takes the gather per pixel below 16 views or so, a plan (whose tables
are there) below fewer, and tiles of 16 instances up to 47 views; the bits are
those of the staged walk, and all are the sum over the views of 64 bits."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from pridediff_amd import load_radontorch
    return load_radontorch()


# width, height, views, batch; instance tile of the plan that walks
CASES = [(301, 340, 1, 1, 1), (301, 340, 15, 2, 2), (301, 340, 16, 1, 1), (520, 501, 9, 3, 4),
         (400, 401, 31, 13, 8), (400, 401, 47, 9, 8), (64, 50, 5, 16, 8), (1030, 1027, 2, 1, 1),
         (1030, 1027, 3, 1, 1)]


@pytest.mark.parametrize("w,h,views,batch,tile", CASES)
@pytest.mark.parametrize("scan,geom", [("para", "ParaDis2d"), ("flat", "FanFlatDis2d"), ("arc", "FanArcDis2d")])
def test_calls_equal_plans(rt, scan, geom, w, h, views, batch, tile):
    pix = 358.4 / max(w, h)
    det = pix * (1.0 if scan == "para" else 1085.6 / 595.0) / (1085.6 if scan == "arc" else 1.0)
    d = int(1.3 * max(w, h))
    g = O.Geom2D(w, h, d, pix, pix, det, 595.0, 1085.6, 0.3, -0.2, 0.1 * det)
    opt = torch.tensor(g.options())
    ang = (np.arange(views) * (2 * np.pi / views) + 0.11).astype(np.float32)
    a = torch.from_numpy(ang).cuda()
    y = torch.rand(batch, 1, views, d, device="cuda",
                   generator=torch.Generator(device="cuda").manual_seed(w + views))
    plan = rt.Plan2d(rt.SCAN[scan], opt, a, batch, tile, -1, 0, 0, 0)
    for name, op, what in ([("ProjTrans", rt.PROJ_T, "proj_t"), ("BackProj", rt.BPROJ, "bproj")] +
                           ([] if scan == "para" else [("BackProjWeighted", rt.BPROJ_W, "bproj_w")])):
        got = getattr(rt, name + geom)(y, opt, a)
        assert torch.equal(got, plan.run(op, y))
        want = O.op2d(scan, what, y[:1, 0].cpu().numpy(), ang, g, "f64")
        err = O.rel_l2(got[:1, 0].cpu().numpy(), want)
        print(f"{scan} {what} {w}x{h}, {views} views, batch {batch}: {err:.2e}", flush=True)
        assert err <= 1e-6  # sums of at most 47 views of FP32 products
