"""ctypes access to the oracle (oracle/liboracle.so) -- the checker of the
tests, never the thing under test."""
from __future__ import annotations

import ctypes
import os
import subprocess

import numpy as np

from cctag_amd import _lib
from tests import golden_tables

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ORACLE_DIR = os.path.join(ROOT, "oracle")
ORACLE_LIB = os.path.join(ORACLE_DIR, "liboracle.so")

_o = None


def load():
    global _o
    if _o is not None:
        return _o
    if not os.path.exists(ORACLE_LIB):
        subprocess.run(["make", "-s", "-C", ORACLE_DIR], check=True)
    o = ctypes.CDLL(ORACLE_LIB)
    vp = ctypes.c_void_p
    o.oracle_front_end.argtypes = [vp, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.POINTER(vp)]
    o.oracle_level_view.argtypes = [vp, ctypes.c_int, ctypes.POINTER(_lib.LevelView)]
    o.oracle_free.argtypes = [vp]
    o.oracle_derivatives.argtypes = [vp, ctypes.c_int, ctypes.c_int, vp, vp]
    o.oracle_derivatives_float.argtypes = [vp, ctypes.c_int, ctypes.c_int, vp, vp]
    o.oracle_canny.argtypes = [vp, vp, ctypes.c_int, ctypes.c_int, ctypes.c_float,
                               ctypes.c_float, vp]
    o.oracle_thin.argtypes = [vp, ctypes.c_int, ctypes.c_int]
    o.oracle_thin_lut.argtypes = [ctypes.c_int, ctypes.c_int]
    o.oracle_downsample.argtypes = [vp, ctypes.c_int, ctypes.c_int, vp, ctypes.c_int, ctypes.c_int]
    o.oracle_bgr_to_gray.argtypes = [vp, ctypes.c_int, ctypes.c_int, ctypes.c_size_t, ctypes.c_int,
                                     vp]
    o.oracle_bgr_to_gray.restype = None
    o.oracle_time_front_end.argtypes = [vp, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    o.oracle_time_front_end.restype = ctypes.c_double
    o.oracle_detect.argtypes = [ctypes.POINTER(_lib.Params), vp, ctypes.c_int, ctypes.c_int,
                                ctypes.POINTER(_lib.Marker), ctypes.c_int]
    o.oracle_detect_threads.argtypes = [ctypes.POINTER(_lib.Params), vp, ctypes.c_int,
                                        ctypes.c_int, ctypes.POINTER(_lib.Marker), ctypes.c_int,
                                        ctypes.c_int]
    o.oracle_grad_cost.argtypes = [vp, ctypes.c_int, ctypes.c_int, vp, vp, ctypes.c_int, ctypes.c_int,
                                   ctypes.c_double, ctypes.c_double, vp, ctypes.POINTER(ctypes.c_int)]
    o.oracle_grad_cost.restype = ctypes.c_double
    o.oracle_time_detect.argtypes = [ctypes.POINTER(_lib.Params), vp, ctypes.c_int,
                                     ctypes.c_int, ctypes.c_int, ctypes.c_int]
    o.oracle_time_detect.restype = ctypes.c_double
    o.oracle_linking_mismatches.argtypes = [vp, ctypes.c_int]
    o.oracle_conic_class_mismatches.argtypes = [vp, ctypes.c_int, ctypes.c_float, ctypes.c_float, vp]
    o.oracle_identify_given.argtypes = [ctypes.POINTER(_lib.Params), vp, ctypes.c_int, ctypes.c_int,
                                        ctypes.POINTER(_lib.IdentMarker), ctypes.c_int,
                                        ctypes.POINTER(_lib.IdentResult)]
    o.oracle_set_bank.argtypes = [ctypes.c_int, vp, ctypes.c_int, ctypes.c_int]
    o.oracle_homography_from_center.argtypes = [vp, ctypes.c_float, ctypes.c_float, vp]
    o.oracle_homography_from_center.restype = None
    o.oracle_conditioner.argtypes = [ctypes.c_float, ctypes.c_float, ctypes.c_float,
                                     ctypes.c_float, vp]
    o.oracle_cut_places.argtypes = [ctypes.c_int, vp, vp, ctypes.c_float, ctypes.c_float, ctypes.c_int,
                                    ctypes.c_int, ctypes.c_int, vp, vp]
    o.oracle_cut_places.restype = None
    o.oracle_sample_cut.argtypes = [vp, ctypes.c_int, ctypes.c_int, vp, vp, ctypes.c_float,
                                    ctypes.c_float, ctypes.c_int, ctypes.c_int, vp]
    o.oracle_conditioner.restype = None
    o.oracle_grid_iterations.argtypes = [ctypes.c_float, ctypes.c_float, ctypes.c_float, ctypes.c_int]
    o.oracle_sorted_outer_points.argtypes = [ctypes.c_float, ctypes.c_float, vp, ctypes.c_int,
                                             ctypes.c_int, vp]
    o.oracle_front_end_params.argtypes = [ctypes.POINTER(_lib.Params), vp, ctypes.c_int,
                                          ctypes.c_int, ctypes.POINTER(vp)]
    o.oracle_edges_and_vote.argtypes = [vp, vp, vp, ctypes.c_int, ctypes.c_int, ctypes.c_int,
                                        ctypes.c_int, ctypes.c_float, ctypes.c_int, ctypes.c_int,
                                        ctypes.POINTER(vp)]
    o.oracle_cut_distances.argtypes = [ctypes.c_int, vp, ctypes.c_int, ctypes.c_float,
                                       ctypes.c_float, vp]
    o.oracle_start_signal.argtypes = [ctypes.c_int]
    o.oracle_start_signal.restype = ctypes.c_float
    o.oracle_refine_stop.argtypes = [vp, ctypes.c_int, ctypes.c_int, vp, ctypes.c_float, ctypes.c_int]
    # the oracle identifies with the reference's own bank tables
    # (CCTagMarkersBank.cpp:120-282, read as data into the golden tables)
    for n, key in ((3, "bank3"), (4, "bank4")):
        b = np.ascontiguousarray(golden_tables.tables()[key], dtype=np.float32)
        if o.oracle_set_bank(n, b.ctypes.data, b.shape[0], b.shape[1]) != 0:
            raise RuntimeError("oracle_set_bank failed")
    _o = o
    return o


def front_end(img: np.ndarray, n_levels: int = 4) -> list:
    """All levels of the oracle front end as dicts (same keys as the product)."""
    o = load()
    img = np.ascontiguousarray(img, dtype=np.uint8)
    h, w = img.shape
    handle = ctypes.c_void_p()
    rc = o.oracle_front_end(img.ctypes.data, w, h, n_levels, ctypes.byref(handle))
    if rc != 0:
        raise RuntimeError("oracle front end failed")
    try:
        out = []
        for l in range(n_levels):
            v = _lib.LevelView()
            o.oracle_level_view(handle, l, ctypes.byref(v))
            out.append(_lib.level_view_to_dict(v))
        return out
    finally:
        o.oracle_free(handle)


def front_end_params(img: np.ndarray, params) -> list:
    """All levels of the oracle front end with the given parameters."""
    o = load()
    img = np.ascontiguousarray(img, dtype=np.uint8)
    h, w = img.shape
    handle = ctypes.c_void_p()
    if o.oracle_front_end_params(ctypes.byref(params), img.ctypes.data, w, h,
                                 ctypes.byref(handle)) != 0:
        raise RuntimeError("oracle front end failed")
    try:
        out = []
        for l in range(params.number_of_processed_multires_layers):
            v = _lib.LevelView()
            o.oracle_level_view(handle, l, ctypes.byref(v))
            out.append(_lib.level_view_to_dict(v))
        return out
    finally:
        o.oracle_free(handle)


def derivatives(img: np.ndarray):
    o = load()
    img = np.ascontiguousarray(img, dtype=np.uint8)
    h, w = img.shape
    dx = np.empty((h, w), np.int16)
    dy = np.empty((h, w), np.int16)
    o.oracle_derivatives(img.ctypes.data, w, h, dx.ctypes.data, dy.ctypes.data)
    return dx, dy


def derivatives_float(img: np.ndarray):
    o = load()
    img = np.ascontiguousarray(img, dtype=np.uint8)
    h, w = img.shape
    dx = np.empty((h, w), np.float32)
    dy = np.empty((h, w), np.float32)
    o.oracle_derivatives_float(img.ctypes.data, w, h, dx.ctypes.data, dy.ctypes.data)
    return dx, dy


def canny(dx: np.ndarray, dy: np.ndarray, low=0.01 * 256, high=0.04 * 256) -> np.ndarray:
    o = load()
    dx = np.ascontiguousarray(dx, np.int16)
    dy = np.ascontiguousarray(dy, np.int16)
    h, w = dx.shape
    e = np.zeros((h, w), np.uint8)
    o.oracle_canny(dx.ctypes.data, dy.ctypes.data, w, h, low, high, e.ctypes.data)
    return e


def thin(edges: np.ndarray) -> np.ndarray:
    o = load()
    e = np.ascontiguousarray(edges, np.uint8).copy()
    h, w = e.shape
    o.oracle_thin(e.ctypes.data, w, h)
    return e


def thin_lut(pass_: int) -> list:
    o = load()
    return [o.oracle_thin_lut(pass_, i) for i in range(512)]


def bgr_to_gray(img: np.ndarray) -> np.ndarray:
    """cv::cvtColor(COLOR_BGR2GRAY) of an h x w x 3 (BGR) or x 4 (BGRA) array."""
    o = load()
    img = np.ascontiguousarray(img, np.uint8)
    h, w, c = img.shape
    out = np.zeros((h, w), np.uint8)
    o.oracle_bgr_to_gray(img.ctypes.data, w, h, ctypes.c_size_t(w * c), c, out.ctypes.data)
    return out


def downsample(img: np.ndarray, size=None) -> np.ndarray:
    """Level.cpp:67 resize to `size` = (w, h), default (w // 2, h // 2)."""
    o = load()
    img = np.ascontiguousarray(img, np.uint8)
    h, w = img.shape
    dw, dh = size if size is not None else (w // 2, h // 2)
    out = np.zeros((dh, dw), np.uint8)
    rc = o.oracle_downsample(img.ctypes.data, w, h, out.ctypes.data, dw, dh)
    if rc != 0:
        raise ValueError("not a shrink")
    return out


def detect(img: np.ndarray, params=None, threads: int = 1) -> list:
    """Full CPU detection (cctagDetection) -> list of marker dicts, sorted by
    id; threads > 1 runs the shared candidate stage on a thread pool."""
    o = load()
    img = np.ascontiguousarray(img, dtype=np.uint8)
    h, w = img.shape
    prm = params if params is not None else _lib.default_params(3)
    buf = (_lib.Marker * 512)()
    n = o.oracle_detect_threads(ctypes.byref(prm), img.ctypes.data, w, h, buf, 512, threads)
    if n < 0:
        raise RuntimeError("oracle detection failed")
    return [buf[i].as_dict() for i in range(min(n, 512))]


def time_detect(img: np.ndarray, iters: int = 1, params=None, threads: int = 1) -> float:
    """Seconds per full CPU detection, averaged over `iters`."""
    o = load()
    img = np.ascontiguousarray(img, dtype=np.uint8)
    h, w = img.shape
    prm = params if params is not None else _lib.default_params(3)
    return o.oracle_time_detect(ctypes.byref(prm), img.ctypes.data, w, h, iters, threads)


def grad_cost(img: np.ndarray, H, stops, n_samples: int = 100, begin: float = 0.25,
              end: float = 1.0, grad: bool = True):
    """Float64 refinement score at homography H (3x3) and, with grad, dC/dH."""
    o = load()
    img = np.ascontiguousarray(img, dtype=np.uint8)
    h, w = img.shape
    Hd = np.ascontiguousarray(np.asarray(H, np.float64).reshape(9))
    st = np.ascontiguousarray(np.asarray(stops, np.float32).reshape(-1, 2))
    g = np.zeros(9, np.float64)
    nv = ctypes.c_int()
    c = o.oracle_grad_cost(img.ctypes.data, w, h, Hd.ctypes.data, st.ctypes.data, len(st), n_samples,
                           begin, end, g.ctypes.data if grad else None, ctypes.byref(nv))
    return c, (g.reshape(3, 3) if grad else None), nv.value


def linking_mismatches(cases: np.ndarray) -> int:
    """Cases (n x 5 float32: front gradient, back gradient, dir) in which the
    candidate stage's linking decisions differ from the float-angle
    expressions."""
    c = np.ascontiguousarray(cases, dtype=np.float32)
    return load().oracle_linking_mismatches(c.ctypes.data, c.shape[0])


def identify_given(img: np.ndarray, markers, params=None) -> list:
    """The oracle's identification of given markers (cctagx_identify's
    counterpart): each a dict with "ellipse" (cx, cy, a, b, angle), "points"
    (n x 4: x, y, gx, gy), "center0" and an optional "scale".  Returns per
    marker a dict: status, id, x, y, quality, homography, stops."""
    o = load()
    img = np.ascontiguousarray(img, dtype=np.uint8)
    h, w = img.shape
    if params is None:
        params = _lib.default_params()
    arr, keep = _lib.ident_markers(markers)
    out = (_lib.IdentResult * max(len(markers), 1))()
    rc = o.oracle_identify_given(ctypes.byref(params), img.ctypes.data, w, h, arr, len(markers), out)
    del keep
    if rc != 0:
        raise RuntimeError("oracle identification failed")
    return [out[i].as_dict() for i in range(len(markers))]


def edges_and_vote(edges: np.ndarray, dx: np.ndarray, dy: np.ndarray, dist_search: int = 30,
                   thr_grad: int = 2500, ratio_voting: float = 4.0, n_crowns: int = 3,
                   min_votes: int = 3) -> dict:
    """Edge points, links, votes and seeds of one level from a given thinned
    edge map {0, 255} and derivative maps (the level-view dict)."""
    o = load()
    e = np.ascontiguousarray(edges, np.uint8)
    gx = np.ascontiguousarray(dx, np.int16)
    gy = np.ascontiguousarray(dy, np.int16)
    h, w = e.shape
    handle = ctypes.c_void_p()
    if o.oracle_edges_and_vote(e.ctypes.data, gx.ctypes.data, gy.ctypes.data, w, h, dist_search,
                               thr_grad, ratio_voting, n_crowns, min_votes,
                               ctypes.byref(handle)) != 0:
        raise RuntimeError("oracle edges_and_vote failed")
    try:
        v = _lib.LevelView()
        o.oracle_level_view(handle, 0, ctypes.byref(v))
        return _lib.level_view_to_dict(v)
    finally:
        o.oracle_free(handle)


def cut_distances(sig, begin: float = 0.25, end: float = 1.0, n_crowns: int = 3) -> np.ndarray:
    """orazioDistanceRobust's distance of one cut signal to every bank row."""
    s = np.ascontiguousarray(sig, np.float32)
    out = np.zeros(256, np.float32)
    n = load().oracle_cut_distances(n_crowns, s.ctypes.data, len(s), begin, end, out.ctypes.data)
    if n < 0:
        raise RuntimeError("oracle cut distances failed")
    return out[:n]


def start_signal(n_crowns: int) -> float:
    return load().oracle_start_signal(n_crowns)


def refine_stop(img: np.ndarray, stop, scale: float = 1.0, n_ref: int = 20):
    """outerEdgeRefinement of one stop (x, y, gx, gy) -> refined (x, y), or
    None when its cut leaves the image."""
    img = np.ascontiguousarray(img, np.uint8)
    h, w = img.shape
    st = np.ascontiguousarray(stop, np.float32).copy()
    ok = load().oracle_refine_stop(img.ctypes.data, w, h, st.ctypes.data, scale, n_ref)
    return (float(st[0]), float(st[1])) if ok else None


def homography_from_center(ellipse, x: float, y: float) -> np.ndarray:
    """The oracle's computeHomographyFromEllipseAndImagedCenter (3 x 3)."""
    e = np.ascontiguousarray(ellipse, np.float32)
    H = np.zeros(9, np.float32)
    load().oracle_homography_from_center(e.ctypes.data, x, y, H.ctypes.data)
    return H.reshape(3, 3)


def conditioner(cx: float, cy: float, a: float, b: float) -> np.ndarray:
    """conditionerFromEllipse after an ellipse with semi-axes a, b set its scale."""
    T = np.zeros(9, np.float32)
    load().oracle_conditioner(cx, cy, a, b, T.ctypes.data)
    return T.reshape(3, 3)


def cut_places(H, stops, n_samples: int, w: int, h: int, begin: float = 0.25, end: float = 1.0):
    """The library's decision for each (homography, stop) -- 0 inside, 1
    outside, 2 unsure -- and the extent (n x 4: min x, max x, min y, max y) of
    the positions at which the cut's samples are read."""
    H = np.ascontiguousarray(np.asarray(H, np.float32).reshape(-1, 9))
    st = np.ascontiguousarray(np.asarray(stops, np.float32).reshape(-1, 2))
    place = np.zeros(len(H), np.int32)
    ext = np.zeros((len(H), 4), np.float32)
    load().oracle_cut_places(len(H), H.ctypes.data, st.ctypes.data, begin, end, n_samples, w, h,
                             place.ctypes.data, ext.ctypes.data)
    return place, ext


def sample_cut(img: np.ndarray, stop, begin: float, end: float, n: int, H=None, start=None):
    """One cut's samples and out-of-bounds flag: through the homography H
    (extractSignalUsingHomography) or, with `start`, straight from start to
    stop (cutInterpolated)."""
    img = np.ascontiguousarray(img, np.uint8)
    h, w = img.shape
    if H is not None:
        m = np.ascontiguousarray(np.asarray(H, np.float32).reshape(9))
    else:
        m = np.zeros(9, np.float32)
        m[:2] = start
    st = np.ascontiguousarray(stop, np.float32)
    sig = np.zeros(n, np.float32)
    oob = load().oracle_sample_cut(img.ctypes.data, w, h, m.ctypes.data, st.ctypes.data, begin, end,
                                   n, int(H is not None), sig.ctypes.data)
    return sig, bool(oob)


def grid_iterations(a: float, b: float, neighbour: float = 0.2, grid_n: int = 5) -> int:
    return load().oracle_grid_iterations(a, b, neighbour, grid_n)


def sorted_outer_points(cx: float, cy: float, pts, requested: int) -> np.ndarray:
    """Indices of the points getSortedOuterPoints keeps, in its order."""
    p = np.ascontiguousarray(np.asarray(pts, np.float32).reshape(-1, 2))
    idx = np.zeros(max(len(p), 1), np.int32)
    n = load().oracle_sorted_outer_points(cx, cy, p.ctypes.data, len(p), requested, idx.ctypes.data)
    return idx[:n]


def conic_class_mismatches(conics: np.ndarray, lo: float = 0.04, hi: float = 25.0):
    """(mismatches, undecided) of the candidate stage's fast RANSAC-trial
    classification against the float derivation, for conics (n x 5 float32)."""
    c = np.ascontiguousarray(conics, dtype=np.float32)
    open_ = ctypes.c_int(0)
    bad = load().oracle_conic_class_mismatches(c.ctypes.data, c.shape[0], lo, hi,
                                               ctypes.byref(open_))
    return bad, open_.value
