"""Uneven batches whose instances hold several slices each (needs an MI355X).

Through the C interface, where an instance's slices share its geometry: every
slice gets the bits of a call of its own, in both directions, for instances
whose bins are staged (tiles of 16 and of 8 rows) and for one whose bins are
too fine.
"""
import ctypes

import numpy as np
import pytest
import torch

from tests.test_zz_no_alloc import LIB, TO_SINO, Geom

pytestmark = pytest.mark.gpu
DD_OK = 0


class Item(ctypes.Structure):
    _fields_ = [("scan", ctypes.c_int), ("geom", Geom), ("views", ctypes.c_int),
                ("batch", ctypes.c_int), ("angles", ctypes.c_void_p),
                ("image_offset", ctypes.c_longlong), ("sino_offset", ctypes.c_longlong)]


@pytest.fixture(scope="module")
def lib():
    import pridediff_amd
    pridediff_amd.load_radontorch()  # libdd binds torch's HIP runtime
    lib = ctypes.CDLL(LIB)
    vp, i, sz = ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t
    for name, res, args in (
            ("dd2d_workspace_size", sz, [i, i, vp, i, i]),
            ("dd2d_run", i, [i, i, vp, vp, vp, vp, i, i, vp, sz, vp]),
            ("dd2d_batch_create", vp, [vp, i]), ("dd2d_batch_device_bytes", sz, [vp]),
            ("dd2d_batch_set_variant", None, [vp, i]), ("dd2d_batch_setup", i, [vp, vp, sz, vp]),
            ("dd2d_batch_run", i, [vp, i, vp, vp, vp]), ("dd2d_batch_destroy", None, [vp])):
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = res, args
    return lib


# width, height, bins, bins per pixel, views, slices
SHAPES = ((61, 33, 97, 1.1, 66, 3), (40, 40, 100, 2.0, 40, 2), (40, 24, 150, 4.0, 24, 5),
          (64, 64, 90, 1.0, 7, 1))


def _batch(lib, scan):
    items, keep, images, sinos = [], [], 0, 0
    for w, h, d, fine, views, slices in SHAPES:
        pix = 358.4 / max(w, h)
        det = pix / fine * (1.0 if scan == 0 else 1085.6 / 595.0) / (1085.6 if scan == 2 else 1.0)
        ang = torch.from_numpy((np.arange(views) * (2 * np.pi / views) + 0.11).astype(np.float32)).cuda()
        g = Geom(w, h, d, pix, pix, det, 595.0, 1085.6, 0.3, -0.2, 0.1 * det)
        items.append(Item(scan, g, views, slices, ang.data_ptr(), images, sinos))
        keep.append(ang)
        images += slices * w * h
        sinos += slices * views * d
    arr = (Item * len(items))(*items)
    b = lib.dd2d_batch_create(arr, len(items))
    assert b
    mem = torch.empty(lib.dd2d_batch_device_bytes(b), dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.dd2d_batch_setup(b, mem.data_ptr(), mem.numel(), stream) == DD_OK
    return b, items, images, sinos, (keep, mem), stream


@pytest.mark.parametrize("scan", [0, 1, 2])
def test_slices_of_an_instance_equal_their_own_calls(lib, scan):
    b, items, images, sinos, keep, stream = _batch(lib, scan)
    gen = torch.Generator(device="cuda").manual_seed(5 + scan)
    try:
        for op in range(4 if scan == 0 else 6):
            print(f"scan {scan} op {op}", flush=True)
            to_sino = op in TO_SINO
            x = torch.rand(images if to_sino else sinos, device="cuda", generator=gen)
            out = torch.full((sinos if to_sino else images,), float("nan"), device="cuda")
            assert lib.dd2d_batch_run(b, op, x.data_ptr(), out.data_ptr(), stream) == DD_OK
            for it in items:
                g, px, bins = it.geom, it.geom.width * it.geom.height, it.views * it.geom.num_det
                n_in, n_out = (px, bins) if to_sino else (bins, px)
                i0, o0 = ((it.image_offset, it.sino_offset) if to_sino
                          else (it.sino_offset, it.image_offset))
                need = lib.dd2d_workspace_size(scan, op, ctypes.byref(g), 1, it.views)
                ws = torch.empty(need, dtype=torch.uint8, device="cuda")
                for k in range(it.batch):
                    one = torch.full((n_out,), float("nan"), device="cuda")
                    src = x[i0 + k * n_in:][:n_in].contiguous()
                    assert lib.dd2d_run(scan, op, ctypes.byref(g), src.data_ptr(), one.data_ptr(),
                                        it.angles, 1, it.views, ws.data_ptr(), need,
                                        stream) == DD_OK
                    assert torch.equal(out[o0 + k * n_out:][:n_out], one), (scan, op, k)
            torch.cuda.synchronize()
    finally:
        lib.dd2d_batch_destroy(b)


@pytest.mark.parametrize("scan", [0, 1, 2])
def test_running_sum_variant_keeps_the_walk_where_bins_are_staged(lib, scan):
    """DD_ADJ_BLOCK_PREFIX: the staged instances' pixels are the walk's bit for
    bit; with finer bins (2 a pixel: staged in parallel beam only) they are
    running sums, within 1e-6 relative L2 of the walk (knots in FP64, one
    rounding to FP32 a view)."""
    b, items, images, sinos, keep, stream = _batch(lib, scan)
    gen = torch.Generator(device="cuda").manual_seed(15 + scan)
    y = torch.rand(sinos, device="cuda", generator=gen)
    try:
        for op in (1, 2):
            got = []
            for variant in (0, 5):
                lib.dd2d_batch_set_variant(b, variant)
                out = torch.full((images,), float("nan"), device="cuda")
                assert lib.dd2d_batch_run(b, op, y.data_ptr(), out.data_ptr(), stream) == DD_OK
                got.append(out)
            for it, (w, h, _, fine, _, k) in zip(items, SHAPES):
                walk, sums = (o[it.image_offset:][:k * w * h] for o in got)
                print(f"scan {scan} op {op} {w}x{h}: {float((walk - sums).norm() / walk.norm()):.2e}",
                      flush=True)
                if fine < 2.0:
                    assert torch.equal(walk, sums)
                else:
                    assert (walk - sums).norm() <= 1e-6 * walk.norm()
            torch.cuda.synchronize()
    finally:
        lib.dd2d_batch_destroy(b)
