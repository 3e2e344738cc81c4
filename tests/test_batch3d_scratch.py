"""Scratch of the sinogram -> volume ops for batches of small volumes, whose
views are split over workgroups: the partial volumes of a batch take 256 MB at
most.  Beyond, a workgroup takes the views' parts one after the other."""
import ctypes
import os

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


class Geom3(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in ("width", "height", "depth", "num_col", "num_row")] + \
               [(n, ctypes.c_float) for n in ("pix_x", "pix_y", "pix_z", "col_size", "row_size",
                                              "iso_source", "source_detector", "shift_x", "shift_y",
                                              "shift_z", "col_shift", "row_shift")]


@pytest.mark.parametrize("batch", [1, 8, 64, 200])
def test_partial_volumes_are_bounded(batch):
    lib = ctypes.CDLL(os.path.join(ROOT, "pridediff_amd", "libdd.so"))
    lib.dd3d_workspace_size.restype = ctypes.c_size_t
    n, views, cols, rows = 128, 90, 180, 160
    g = Geom3(n, n, n, cols, rows, 1.0, 1.0, 1.0, 1.5, 1.5, 1000.0, 1500.0, 0, 0, 0, 0, 0)
    size = lib.dd3d_workspace_size(3, 1, ctypes.byref(g), batch, views)
    sino = 4 * views * cols * rows * (-(-batch // 4) * 4 if batch > 2 else batch)
    tables = 16 << 20
    assert sino < size <= sino + tables + (256 << 20)


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [11, 19])
def test_parts_one_after_the_other_keep_the_bits(batch):
    """96^3 x 72 views are split in 9 parts, 32 MB an instance: the parts of a
    batch of 4 fit, those of 11 and 19 do not.  Every volume is the one of a
    batch of 4, bit for bit."""
    from pridediff_amd import load_radontorch
    rt = load_radontorch()
    n, views = 96, 72
    opt = torch.tensor([n, n, n, 140, 120, 1.0, 1.0, 1.0, 1.5, 1.5, 1000.0, 1500.0, 0.1, -0.2, 0.3,
                        0.2, 0.1])
    ang = torch.arange(views, device="cuda", dtype=torch.float32) * (2 * np.pi / views)
    gen = torch.Generator(device="cuda").manual_seed(batch)
    y = torch.rand(batch, 1, views, 120, 140, device="cuda", generator=gen)
    got = rt.ProjTransConeFlatDis3d(y, opt, ang)
    for b in range(0, batch, 4):
        few = torch.zeros(4, 1, views, 120, 140, device="cuda")
        few[:min(4, batch - b)] = y[b:b + 4]
        assert torch.equal(rt.ProjTransConeFlatDis3d(few, opt, ang)[:min(4, batch - b)], got[b:b + 4])
