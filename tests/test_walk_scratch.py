"""Memory of the 2D sinogram -> image ops where the bins are too fine to be
staged: neither the staged walk's range table nor its partial images (host
queries, no GPU)."""
import ctypes
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


class Geom(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in ("width", "height", "num_det")] + \
               [(n, ctypes.c_float) for n in ("pix_x", "pix_y", "det", "iso_source",
                                              "source_detector", "shift_x", "shift_y", "bin_shift")]


@pytest.mark.parametrize("batch", [1, 16])
@pytest.mark.parametrize("scan", [0, 1, 2])
def test_fine_bins_take_no_walk_tables(scan, batch):
    lib = ctypes.CDLL(os.path.join(ROOT, "pridediff_amd", "libdd.so"))
    for fn in ("dd2d_workspace_size", "dd2d_geometry_size", "dd2d_planned_workspace_size"):
        getattr(lib, fn).restype = ctypes.c_size_t
    n, views, fine = 512, 180, 4.0
    pix = 0.7
    det = pix / fine * (1.0 if scan == 0 else 1085.6 / 595.0) / (1085.6 if scan == 2 else 1.0)
    d = 2240
    g = Geom(n, n, d, pix, pix, det, 595.0, 1085.6, 0, 0, 0)
    tables = views * (96 + 8 * (d + 1) + 4 * d + 16 * n + 4 * n)
    sino = 4 * views * d * batch
    spare = 8 << 10  # alignment
    for op in (1, 2) + ((4,) if scan else ()):
        assert lib.dd2d_workspace_size(scan, op, ctypes.byref(g), batch, views) <= tables + sino + spare
    assert lib.dd2d_geometry_size(scan, ctypes.byref(g), views) <= tables + spare
    # a plan at instance tile 1 also holds the running sums' buffers
    if batch == 16:
        assert lib.dd2d_planned_workspace_size(scan, 1, ctypes.byref(g), batch, views, 16) <= sino + spare
