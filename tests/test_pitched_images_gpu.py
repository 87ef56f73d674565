"""Images whose rows lie apart (stride > width) through the refiner and the
allocation-free grid search: the same results as their packed copies, from
strides that fit the device's room for the image as they lie and from those
that do not."""
import ctypes

import numpy as np
import pytest

from cctag_amd import _lib, synth
from cctag_amd.detector import Refiner

STATIC_PIXELS = 1920 * 1088


def static_grid(base, w, h, stride, markers):
    lib = _lib.load()
    arr = (_lib.RefineMarker * len(markers))()
    for i, m in enumerate(markers):
        arr[i].ellipse[:] = [float(v) for v in m["ellipse"]]
        arr[i].center0[:] = [float(v) for v in m["center0"]]
        arr[i].n_cuts = len(m["stops"])
        for k, (x, y) in enumerate(np.asarray(m["stops"], np.float32)):
            arr[i].stops[k][0], arr[i].stops[k][1] = float(x), float(y)
    c, ok = np.zeros((len(markers), 2), np.float32), np.zeros(len(markers), np.int32)
    _lib.check(lib.cctagx_refine_grid_static(ctypes.byref(_lib.default_params(3)), base.ctypes.data, w, h,
                                             stride, arr, len(markers), c.ctypes.data, ok.ctypes.data),
               "cctagx_refine_grid_static")
    return c.tobytes(), ok.tobytes()


@pytest.mark.gpu
@pytest.mark.parametrize("extra", [0, 1, 37, 4000, 30000])
def test_rows_apart(extra):
    img, ms = synth.refine_mosaic(9, unique=9, seed=3)
    h, w = img.shape
    assert (h - 1) * (w + 30000) + w > STATIC_PIXELS > (h - 1) * (w + 37) + w
    base = np.random.default_rng(extra).integers(0, 256, (h, w + extra), dtype=np.uint8)
    base[:, :w] = img
    base = base.ravel()[:(h - 1) * (w + extra) + w].copy()  # nothing after the last row
    want = static_grid(img, w, h, w, ms)
    print("rows apart", extra, flush=True)
    assert static_grid(base, w, h, w + extra, ms) == want
    with Refiner(len(ms)) as r:
        got = []
        for data, stride in ((img, w), (base, w + extra)):
            _lib.check(r._lib.cctagx_refiner_set_image(r._h, data.ctypes.data, w, h, stride), "set_image")
            r.set_markers(ms)
            c, ok = r.grid()
            got.append((c.tobytes(), ok.astype(np.int32).tobytes()))
    assert got[0] == got[1] == want
