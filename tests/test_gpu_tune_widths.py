"""The tuner sweeps the per-pixel adjoint's workgroup width only where that
gather runs (needs an MI355X)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("num_det,det,views,gather", [(180, 1.2858 * 4, 40, False),
                                                      (700, 1.2858, 40, True),
                                                      (180, 1.2858 * 4, 7, True)])
def test_widths_swept_where_they_reach_a_kernel(num_det, det, views, gather):
    """128 x 128 pixels: about one bin a pixel (staged), four (too fine), and
    few views."""
    from pridediff_amd import load_radontorch
    from pridediff_amd.autotune import tune_uniform
    from pridediff_amd.deeprecon.torch.projector import projector2d
    rt = load_radontorch()
    P = projector2d(128, num_det, 0.7 * 4, det, 595.0, 1085.6, scan_type="arc").cuda()
    ang = (torch.arange(views, device="cuda", dtype=torch.float32) * (2 * np.pi / views))
    info = {}
    tuned = tune_uniform(P, ang, 2, tiles=(2,), use_cache=False, report=info, running_sums=False)
    assert any("/pix" in k for k in info["swept"]) == gather
    assert tuned.plan.pixel_gather(rt.PROJ_T) == gather
    assert gather or info["shape"][2] == 0
    assert not tuned.plan.pixel_gather(rt.PROJ)
