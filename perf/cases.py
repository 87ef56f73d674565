"""The work that users of this framework have it do, as timed cases.

A case names an entry point and the sizes it runs at; prepare() makes what a
user's program has in hand before the call (host frames, since cameras and
decoders deliver those, or a refiner holding its image and markers), run() is
one call, exact() the same result in 64 bits where the call computes numbers
rather than takes decisions.

Frames follow the synthetic configurations of cctag_amd/synth.py (markers drawn
through a plane-to-image homography over gradient noise, blur, sensor noise),
rendered with torch so that they are quick to make.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cctag_amd import _lib, synth
from cctag_amd.bank import bank_ratios
from cctag_amd.detector import BatchDetector, Detector, Refiner

DEV = "cuda" if torch.cuda.is_available() else "cpu"
N_SAMPLES = 100        # samples along a cut (the default parameters)
GRID = 5               # grid points per axis of the centre search
NEIGHBOUR = 0.2        # its first neighbourhood, in outer semi-axes
BEGIN = {3: 0.25, 4: 0.26}  # where a cut's samples begin, in outer radii
TILE = 160             # tile of the refinement mosaic, pixels


# --------------------------------------------------------------------------
# the cases

def listed():
    def detect(name, w, h, markers, **kw):
        c = {"name": name, "op": "detect", "width": w, "height": h, "markers": markers,
             "channels": 1, "crowns": 3, "rmin": 25.0, "rmax": 200.0, "tilt": 60.0,
             "blur": 2.0, "noise": 6.0, "occluded": 0.2, "distractors": 0, "motion": 0.0}
        return {**c, **kw}

    return [
        # one small camera frame with two markers: the smallest detection, where latency counts
        detect("detect_640x480", 640, 480, 2, rmin=30.0, rmax=70.0, tilt=45.0),
        # a 720p video frame with four-ring markers (the 128-row bank)
        detect("detect_1280x720_4crowns", 1280, 720, 6, crowns=4, rmin=40.0, rmax=120.0, tilt=45.0,
               blur=1.0, noise=4.0, occluded=0.0),
        # a decoded color frame of a laptop camera: converted on the device, and of a size whose
        # pyramid levels are not exact halves
        detect("detect_bgr_1366x768", 1366, 768, 8, channels=3, rmax=110.0),
        # the ordinary frame: full HD, sixteen markers
        detect("detect_1920x1080", 1920, 1080, 16),
        # a cluttered 4K frame: the largest single detection
        detect("detect_3840x2160", 3840, 2160, 32, rmin=15.0, rmax=400.0, tilt=70.0, blur=1.0,
               noise=8.0, occluded=0.0, distractors=200, motion=7.0),
        # images of several cameras taken together, of uneven sizes
        {"name": "batch_uneven_16", "op": "batch", "gradient": 0, "markers": 12, "distractors": 40,
         "sizes": "640x480*5 1280x720*4 1001x751*1 1920x1080*4 3840x2160*2"},
        # full HD frames of one video, their centres refined by descent
        {"name": "batch_gradient_1080p_8", "op": "batch", "gradient": 30, "markers": 16,
         "distractors": 0, "sizes": "1920x1080*8"},
        # tracking: markers predicted from the frame before are identified on a new frame
        {"name": "identify_1920x1080", "op": "identify", "width": 1920, "height": 1080,
         "markers": 16},
        # a serving loop that must not allocate: a few markers of one small image
        {"name": "static_grid_8", "op": "static", "markers": 8, "cuts": 22, "steps": 0},
        # centre search of the markers of many images at once
        {"name": "refiner_grid_1024", "op": "grid", "markers": 1024, "cuts": 22, "steps": 0},
        # the same by the differentiable score, the largest refinement
        {"name": "refiner_refine_4096", "op": "refine", "markers": 4096, "cuts": 22, "steps": 20},
        # the score and its gradient, forward and adjoint, for a caller's own optimizer
        {"name": "refiner_cost_grad_2048", "op": "cost_grad", "markers": 2048, "cuts": 22,
         "steps": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Frames from 320x240 to 3840x2160 of any aspect and parity, gray or color, three or four
    crowns; batches of 2 to 16 frames; refinements of 1 to 4096 markers with 8 to 32 cuts."""
    op = rng.choice(["detect", "detect", "detect", "batch", "identify", "static", "grid", "refine",
                     "cost_grad"])
    if op == "detect":
        h = _log_int(rng, 240, 2160)
        w = min(3840, int(h * rng.uniform(1.2, 1.8)))
        crowns = rng.choice([3, 3, 4])
        return {"op": op, "width": w, "height": h, "markers": rng.randint(1, max(1, min(32, h // 60))),
                "channels": rng.choice([1, 1, 3, 4]), "crowns": crowns,
                "rmin": 25.0 if crowns == 3 else 35.0, "rmax": round(0.18 * h, 1),
                "tilt": round(rng.uniform(20.0, 65.0), 1), "blur": round(rng.uniform(0.8, 2.0), 2),
                "noise": round(rng.uniform(2.0, 8.0), 2), "occluded": rng.choice([0.0, 0.2]),
                "distractors": rng.randint(0, h // 20), "motion": 0.0}
    if op == "batch":
        sizes = ["%dx%d" % (min(3840, int(h * 1.6) + rng.randint(0, 5)), h)
                 for h in (_log_int(rng, 300, 1200) for _ in range(rng.randint(2, 16)))]
        return {"op": op, "gradient": rng.choice([0, 0, 30]), "markers": rng.randint(2, 16),
                "distractors": rng.randint(0, 60), "sizes": " ".join(s + "*1" for s in sizes)}
    if op == "identify":
        h = _log_int(rng, 480, 2160)
        return {"op": op, "width": min(3840, int(h * 1.7)), "height": h,
                "markers": rng.randint(1, 32)}
    cuts = rng.randint(8, 32)
    return {"op": op, "cuts": cuts, "steps": rng.randint(5, 20) if op == "refine" else 0,
            "markers": rng.randint(1, 64) if op == "static" else _log_int(rng, 1, 4096 * 22 // max(cuts, 22))}


# --------------------------------------------------------------------------
# synthetic frames

def _rngs(seed):
    return np.random.default_rng(seed), torch.Generator(device=DEV).manual_seed(seed)


def _background(h, w, amp, gen, cell=256):
    """Gradient noise of amplitude amp around mid gray."""
    gh, gw = h // cell + 2, w // cell + 2
    ang = torch.rand((gh, gw), generator=gen, device=DEV) * (2 * math.pi)
    gx, gy = torch.cos(ang), torch.sin(ang)
    y = (torch.arange(h, device=DEV) + 0.5) / cell
    x = (torch.arange(w, device=DEV) + 0.5) / cell
    yi, xi = y.long(), x.long()
    fy, fx = (y - yi)[:, None], (x - xi)[None, :]

    def corner(dy, dx):
        iy, ix = (yi + dy)[:, None], (xi + dx)[None, :]
        return gx[iy, ix] * (fx - dx) + gy[iy, ix] * (fy - dy)

    def fade(t):
        return t * t * t * (t * (t * 6 - 15) + 10)

    u, v = fade(fx), fade(fy)
    top = corner(0, 0) + u * (corner(0, 1) - corner(0, 0))
    bottom = corner(1, 0) + u * (corner(1, 1) - corner(1, 0))
    return 128.0 + amp * math.sqrt(2.0) * (top + v * (bottom - top))


def _draw_marker(img, H, ratios, ss=3):
    """One marker and its white quiet zone (to 1.4 outer radii), ss x ss samples per pixel."""
    h, w = img.shape
    t = np.linspace(0, 2 * np.pi, 128, endpoint=False)
    q = H @ np.stack([1.42 * np.cos(t), 1.42 * np.sin(t), np.ones_like(t)])
    qx, qy = q[0] / q[2], q[1] / q[2]
    x0, x1 = max(int(qx.min()) - 1, 0), min(int(qx.max()) + 2, w)
    y0, y1 = max(int(qy.min()) - 1, 0), min(int(qy.max()) + 2, h)
    if x0 >= x1 or y0 >= y1:
        return
    Hi = np.linalg.inv(H)
    xs = x0 + (torch.arange((x1 - x0) * ss, device=DEV) + 0.5)[None, :] / ss
    ys = y0 + (torch.arange((y1 - y0) * ss, device=DEV) + 0.5)[:, None] / ss
    u, v, k = (float(r[0]) * xs + float(r[1]) * ys + float(r[2]) for r in Hi)
    rho = torch.sqrt(u * u + v * v) / k.abs()
    rings = torch.zeros_like(rho, dtype=torch.int32)
    for r in ratios:
        rings += (rho >= 1.0 / float(r)).int()
    val = torch.where((rings % 2 == 0) | (rho >= 1.0), synth.WHITE, synth.BLACK)
    inside = (rho <= 1.4).float()

    def pool(a):
        return a.reshape(y1 - y0, ss, x1 - x0, ss).mean(dim=(1, 3))

    cov = pool(inside)
    img[y0:y1, x0:x1] = img[y0:y1, x0:x1] * (1 - cov) + pool(val * inside)


def _draw_distractor(img, rng, rmin, rmax):
    """A filled ellipse or an elliptical ring of random gray."""
    h, w = img.shape
    a = rng.uniform(rmin, rmax)
    b, cx, cy = a * rng.uniform(0.3, 1.0), rng.uniform(0, w), rng.uniform(0, h)
    ang, level, thick = rng.uniform(0, np.pi), rng.uniform(10, 245), rng.uniform(0.08, 0.3)
    ring = rng.random() < 0.5
    x0, x1 = max(int(cx - a) - 2, 0), min(int(cx + a) + 3, w)
    y0, y1 = max(int(cy - a) - 2, 0), min(int(cy + a) + 3, h)
    if x0 >= x1 or y0 >= y1:
        return
    X = torch.arange(x0, x1, device=DEV)[None, :] + 0.5 - cx
    Y = torch.arange(y0, y1, device=DEV)[:, None] + 0.5 - cy
    c, s = math.cos(ang), math.sin(ang)
    r = torch.sqrt(((c * X + s * Y) / a) ** 2 + ((c * Y - s * X) / b) ** 2)
    cov = ((1.0 - r) * b + 0.5).clamp(0, 1)  # about one pixel of edge
    if ring:
        cov = cov * ((r - (1.0 - thick)) * b + 0.5).clamp(0, 1)
    img[y0:y1, x0:x1] = img[y0:y1, x0:x1] * (1 - cov) + level * cov


def _shift_sum(img, taps):
    """Sum of weighted copies of img moved by (dy, dx), the border repeated."""
    r = max(max(abs(dy), abs(dx)) for dy, dx, _ in taps)
    h, w = img.shape
    p = torch.nn.functional.pad(img[None, None], (r, r, r, r), mode="replicate")[0, 0]
    out = torch.zeros_like(img)
    for dy, dx, wt in taps:
        out += wt * p[r + dy:r + dy + h, r + dx:r + dx + w]
    return out


def _blur(img, sigma):
    n = max(1, int(math.ceil(3 * sigma)))
    k = [math.exp(-0.5 * (i / sigma) ** 2) for i in range(-n, n + 1)]
    k = [v / sum(k) for v in k]
    img = _shift_sum(img, [(i - n, 0, v) for i, v in enumerate(k)])
    return _shift_sum(img, [(0, i - n, v) for i, v in enumerate(k)])


def _motion(img, length, angle):
    taps, n = {}, 33
    for t in np.linspace(-length / 2, length / 2, n):
        at = (int(round(t * math.sin(angle))), int(round(t * math.cos(angle))))
        taps[at] = taps.get(at, 0.0) + 1.0 / n
    return _shift_sum(img, [(dy, dx, v) for (dy, dx), v in taps.items()])


def _frame(w, h, markers, seed, crowns=3, rmin=25.0, rmax=200.0, tilt=60.0, blur=2.0, noise=6.0,
           occluded=0.0, distractors=0, motion=0.0, channels=1):
    """A uint8 frame (numpy) and the homographies of its markers."""
    rng, gen = _rngs(seed)
    img = _background(h, w, 20.0, gen)
    for _ in range(distractors):
        _draw_distractor(img, rng, 5.0, min(300.0, 0.25 * h))
    ratios, placed, Hs = bank_ratios(crowns), [], []
    for _ in range(markers):
        r = rng.uniform(rmin, max(rmin, min(rmax, 0.3 * min(w, h))))
        for attempt in range(200):
            if attempt and attempt % 40 == 0:
                r = max(rmin, r * 0.8)
            rb = min(1.5 * r, 0.49 * min(w, h))
            x, y = rng.uniform(rb, w - rb), rng.uniform(rb, h - rb)
            if all(math.hypot(x - px, y - py) > rb + pr for px, py, pr in placed):
                break
        else:
            continue
        H = synth.marker_homography(x, y, r, math.radians(rng.uniform(0, tilt)),
                                    rng.uniform(0, 2 * np.pi), rng.uniform(0, 2 * np.pi),
                                    2.0 * max(w, h))
        _draw_marker(img, H, ratios[int(rng.integers(0, len(ratios)))])
        placed.append((x, y, rb))
        Hs.append(H)
        if rng.random() < occluded:
            phi, half = rng.uniform(0, 2 * np.pi), rng.uniform(0.15, 0.3) * r
            p = H @ np.array([math.cos(phi), math.sin(phi), 1.0])
            ox, oy = p[0] / p[2], p[1] / p[2]
            img[max(int(oy - half), 0):max(int(oy + half), 0),
                max(int(ox - half), 0):max(int(ox + half), 0)] = 25.0
    img = _blur(img, rng.uniform(0.5, max(0.6, blur)))
    if motion > 0:
        img = _motion(img, rng.uniform(1.0, motion), rng.uniform(0, np.pi))
    if channels > 1:  # a color cast per channel; alpha, where there is one, is opaque
        cast = torch.tensor([0.92, 1.0, 0.97], device=DEV)
        img = img[:, :, None] * cast
    img = img + noise * torch.randn(img.shape, generator=gen, device=DEV)
    img = img.round().clamp(0, 255).to(torch.uint8)
    if channels == 4:
        img = torch.cat([img, torch.full((h, w, 1), 255, dtype=torch.uint8, device=DEV)], dim=2)
    return np.ascontiguousarray(img.cpu().numpy()), Hs


def _mosaic(n, cuts, seed, unique=64):
    """n markers of 20 to 36 px radius seen under strong perspective, one to a tile."""
    rng, gen = _rngs(seed)
    ratios, tiles, Hs = bank_ratios(3), [], []
    for _ in range(min(unique, n)):
        r = rng.uniform(20.0, 36.0)
        c = TILE / 2 + rng.uniform(-3, 3, size=2)
        H = synth.marker_homography(c[0], c[1], r, math.radians(rng.uniform(0, 60)),
                                    rng.uniform(0, 2 * np.pi), rng.uniform(0, 2 * np.pi),
                                    r * rng.uniform(4.0, 8.0))
        t = torch.full((TILE, TILE), 128.0, device=DEV)
        _draw_marker(t, H, ratios[int(rng.integers(0, len(ratios)))])
        tiles.append(_blur(t, rng.uniform(0.5, 1.5)))
        Hs.append(H)
    side = int(math.ceil(math.sqrt(n)))
    order = torch.arange(side * side, device=DEV) % len(tiles)
    img = torch.stack(tiles)[order].reshape(side, side, TILE, TILE).permute(0, 2, 1, 3)
    img = img.reshape(side * TILE, side * TILE)
    img = img + 6.0 * torch.randn(img.shape, generator=gen, device=DEV)
    img = img.round().clamp(0, 255).to(torch.uint8).cpu().numpy()
    markers = []
    for k in range(n):
        ty, tx = divmod(k, side)
        T = np.array([[1.0, 0.0, tx * TILE], [0.0, 1.0, ty * TILE], [0.0, 0.0, 1.0]])
        markers.append(synth.refine_marker(T @ Hs[k % len(Hs)], cuts))
    return np.ascontiguousarray(img), markers


def _sizes(case):
    out = []
    for part in case["sizes"].split():
        size, times = part.split("*")
        w, h = size.split("x")
        out += [(int(w), int(h))] * int(times)
    return out


def _tracked(H):
    """A marker as a tracker hands it over: its outer ellipse and the edge points around it with
    their gradients (outwards: the outer ring is black on white)."""
    D = synth.DETECTOR_SHIFT @ H
    e = synth.ellipse_of(D)
    n = max(40, int(4 * (e[2] + e[3])))
    t = 2 * np.pi * np.arange(n) / n
    p = D @ np.stack([np.cos(t), np.sin(t), np.ones(n)])
    p = (p[:2] / p[2]).T
    c, s = math.cos(e[4]), math.sin(e[4])
    u, v = c * (p[:, 0] - e[0]) + s * (p[:, 1] - e[1]), c * (p[:, 1] - e[1]) - s * (p[:, 0] - e[0])
    g = np.stack([c * u / e[2] ** 2 - s * v / e[3] ** 2, s * u / e[2] ** 2 + c * v / e[3] ** 2], 1)
    g = 100.0 * g / np.linalg.norm(g, axis=1, keepdims=True)
    return {"ellipse": e, "center0": (e[0], e[1]), "scale": 1.0,
            "points": np.concatenate([np.rint(p), np.rint(g)], 1).astype(np.float32)}


# --------------------------------------------------------------------------
# prepare and run

def prepare(case, seed):
    op = case["op"]
    if op == "detect":
        keys = ("crowns", "rmin", "rmax", "tilt", "blur", "noise", "occluded", "distractors",
                "motion", "channels")
        img, _ = _frame(case["width"], case["height"], case["markers"], seed,
                        **{k: case[k] for k in keys})
        return {"op": op, "img": img, "color": case["channels"] > 1,
                "rows": 64 + 8 * case["markers"],
                "det": Detector(case["width"], case["height"], n_crowns=case["crowns"])}
    if op == "batch":
        sizes = _sizes(case)
        imgs = [_frame(w, h, case["markers"], seed * 1000 + k, rmax=0.16 * h, occluded=0.2,
                       distractors=case["distractors"])[0] for k, (w, h) in enumerate(sizes)]
        b = BatchDetector(sizes)
        b.set_refinement(case["gradient"])
        return {"op": op, "imgs": imgs, "batch": b,
                "rows": 64 + 8 * case["markers"] * len(sizes)}
    if op == "identify":
        img, Hs = _frame(case["width"], case["height"], case["markers"], seed)
        return {"op": op, "img": img, "det": Detector(case["width"], case["height"]),
                "markers": [_tracked(H) for H in Hs], "rows": case["markers"]}
    img, markers = _mosaic(case["markers"], case["cuts"], seed)
    if op == "static":
        arr = (_lib.RefineMarker * len(markers))()
        for a, m in zip(arr, markers):
            a.ellipse[:], a.center0[:], a.n_cuts = m["ellipse"], m["center0"], len(m["stops"])
            for k, (x, y) in enumerate(m["stops"]):
                a.stops[k][:] = (float(x), float(y))
        return {"op": op, "img": img, "markers": arr, "n": len(markers),
                "params": _lib.default_params(3), "lib": _lib.load()}
    r = Refiner(len(markers))
    r.set_image(img)
    r.set_markers(markers)
    return {"op": op, "ref": r, "steps": case["steps"], "H": _homographies(markers, seed)}


def _homographies(markers, seed):
    """Where a caller's optimizer stands: near the true homographies."""
    rng = np.random.default_rng(seed + 77)
    H = np.stack([m["H"] for m in markers])
    T = np.tile(np.eye(3), (len(H), 1, 1))
    T[:, :2, 2] = rng.normal(0.0, 0.02, size=(len(H), 2))  # marker-plane shift of the centre
    H = H @ T
    return (H / H[:, 2:, 2:]).reshape(-1, 9).astype(np.float32)


def _rows(values, rows, *shape, dtype=np.float32):
    """values as the first rows of an array of a size that does not depend on how many there are."""
    out = np.zeros((rows, *shape), dtype)
    if values:
        out[:len(values)] = values
    return out


def _marker_arrays(markers, rows):
    return {"count": len(markers),
            "id": _rows([(m["id"], m["status"], m["pyramid_level"]) for m in markers], rows, 3,
                        dtype=np.int32),
            "center": _rows([(m["x"], m["y"]) for m in markers], rows, 2),
            "quality": _rows([m["quality"] for m in markers], rows),
            "ellipse": _rows([m["ellipse"] for m in markers], rows, 5),
            "homography": _rows([m["homography"] for m in markers], rows, 9)}


def run(s):
    op = s["op"]
    if op == "detect":
        return _marker_arrays(s["det"].detect_bgr(s["img"]) if s["color"]
                              else s["det"].detect(s["img"]), s["rows"])
    if op == "batch":
        for f, img in enumerate(s["imgs"]):
            s["batch"].load(f, img)
        frames = s["batch"].detect()
        out = _marker_arrays([m for f in frames for m in f], s["rows"])
        out["per_frame"] = np.array([len(f) for f in frames], np.int32)
        return out
    if op == "identify":
        s["det"].front_end(s["img"])
        got = s["det"].identify(s["markers"])
        n = s["rows"]
        stops = np.zeros((n, 32, 2), np.float32)
        for k, m in enumerate(got):
            stops[k, :len(m["stops"])] = m["stops"]
        return {"id": _rows([(m["id"], m["status"]) for m in got], n, 2, dtype=np.int32),
                "center": _rows([(m["x"], m["y"]) for m in got], n, 2),
                "quality": _rows([m["quality"] for m in got], n),
                "homography": _rows([m["homography"] for m in got], n, 9), "stops": stops}
    if op == "static":
        c, ok = np.zeros((s["n"], 2), np.float32), np.zeros(s["n"], np.int32)
        h, w = s["img"].shape
        _lib.check(s["lib"].cctagx_refine_grid_static(
            s["params"], s["img"].ctypes.data, w, h, s["img"].strides[0], s["markers"], s["n"],
            c.ctypes.data, ok.ctypes.data), "cctagx_refine_grid_static")
        return {"center": c, "ok": ok}
    if op == "grid":
        c, ok = s["ref"].grid()
        return {"center": c, "ok": ok.astype(np.int32)}
    if op == "refine":
        c, cost = s["ref"].refine(s["steps"])
        return {"center": c, "cost": cost}
    cost, grad = s["ref"].cost_grad(s["H"])
    return {"cost": cost, "grad": grad}


# --------------------------------------------------------------------------
# what a pass cannot do without

def _iterations(semi_axis):
    ns, it = NEIGHBOUR, 0
    while ns * semi_axis > 0.02:
        ns, it = ns / 2, it + 1
    return it


def work(case):
    """Bytes: frames and markers in, results out, each once.  Operations: the two 72-tap
    derivative filters over the pyramid and, per marker, the centre search: 25 per cut sample, 3
    per sample and pair of cuts (the descent: forward and adjoint, 75 per sample and step)."""
    op, n = case["op"], case["markers"]
    if op in ("detect", "identify", "batch"):
        sizes = _sizes(case) if op == "batch" else [(case["width"], case["height"])]
        pix = sum(w * h for w, h in sizes)
        marker = GRID * GRID * 10 * (22 * N_SAMPLES * 25 + N_SAMPLES * 3 * 22 * 21 // 2)
        return {"bytes": pix * case.get("channels", 1) + 84 * n * len(sizes),
                "flops": pix * 1.33 * 288 + n * len(sizes) * marker}
    cuts = case["cuts"]
    samples = cuts * N_SAMPLES
    score = samples * 25 + N_SAMPLES * 3 * cuts * (cuts - 1) // 2
    quads = samples * 2  # image bytes near the cuts, the disc read once
    if op == "cost_grad":
        return {"bytes": n * (36 + 88 + 32 + 8 * cuts + quads), "flops": n * samples * 75}
    if op == "refine":
        return {"bytes": n * (16 + 32 + 8 * cuts + quads),
                "flops": n * (GRID * GRID * score + case["steps"] * samples * 75)}
    side = int(math.ceil(math.sqrt(n))) * TILE
    frame = side * side if op == "static" else n * quads
    return {"bytes": frame + n * (12 + 32 + 8 * cuts),
            "flops": n * GRID * GRID * _iterations(30.0) * score}


# --------------------------------------------------------------------------
# the same in 64 bits

def _sample(img, w, x, y):
    """Half the bilinear value of the uint8 image at (x, y)."""
    ix, iy = x.detach().long(), y.detach().long()
    fx, fy = x - ix, y - iy
    at = iy * w + ix

    def px(o):
        return img[at + o].double()

    return 0.5 * ((px(0) * (1 - fx) + px(1) * fx) * (1 - fy) + (px(w) * (1 - fx) + px(w + 1) * fx) * fy)


def _score(s):
    """Mean over pairs of cuts of the summed squared differences; s: (..., cuts, samples)."""
    m = s.shape[-2]
    per = m * (s * s).sum(-2) - s.sum(-2) ** 2
    return per.sum(-1) / (0.5 * m * (m - 1))


def _positions(t, begin):
    return torch.tensor(begin, device=t.device, dtype=torch.float64) + torch.arange(
        N_SAMPLES, device=t.device, dtype=torch.float64) * ((1.0 - begin) / (N_SAMPLES - 1))


def _center_score(img, w, conic, stops, c):
    """The score of imaged centres c (n, 2).  The polar of the centre is the marker plane's
    vanishing line, which gives the weights of the projective segment centre -> stop."""
    one = torch.ones_like(c[:, :1])
    line = torch.einsum("nij,nj->ni", conic, torch.cat([c, one], 1))
    wc = 1.0 / (line[:, :2] * c).sum(1).add(line[:, 2])                        # n
    wp = 1.0 / (torch.einsum("nj,nkj->nk", line[:, :2], stops) + line[:, 2:])  # n, k
    t = _positions(c, BEGIN[3])
    a = (t * wp[:, :, None])                       # n, k, i
    b = (1.0 - t)[None, None, :] * wc[:, None, None]
    x = (a * stops[:, :, None, 0] + b * c[:, None, None, 0]) / (a + b)
    y = (a * stops[:, :, None, 1] + b * c[:, None, None, 1]) / (a + b)
    return _score(_sample(img, w, x, y))


def _conics(markers, device):
    out = []
    for m in markers:
        cx, cy, a, b, ang = (float(np.float32(v)) for v in m["ellipse"])
        c, s = math.cos(ang), math.sin(ang)
        M = np.array([[c / a, s / a, -(c * cx + s * cy) / a], [-s / b, c / b, (s * cx - c * cy) / b],
                      [0.0, 0.0, 1.0]])
        out.append(M.T @ np.diag([1.0, 1.0, -1.0]) @ M)
    return torch.tensor(np.stack(out), device=device, dtype=torch.float64)


def exact(case, seed):
    op = case["op"]
    if op in ("detect", "batch", "identify"):
        return None  # decisions: which edges, ellipses and cuts are kept
    img, markers = _mosaic(case["markers"], case["cuts"], seed)
    w = img.shape[1]
    flat = torch.from_numpy(img).to(DEV).reshape(-1)
    parts = []
    for k in range(0, len(markers), 512):
        ms = markers[k:k + 512]
        f32 = lambda key: torch.tensor(  # noqa: E731
            np.stack([np.asarray(m[key], np.float32) for m in ms]), device=DEV).double()
        stops = f32("stops")
        if op == "cost_grad":
            H = torch.from_numpy(_homographies(markers, seed)[k:k + 512]).to(DEV).double()
            parts.append(_exact_grad(flat, w, H.reshape(-1, 3, 3), stops))
        else:
            parts.append(_exact_search(flat, w, _conics(ms, DEV), stops, f32("center0"),
                                       [max(m["ellipse"][2:4]) for m in ms], op, case["steps"]))
    out = [torch.cat(p).cpu().numpy() for p in zip(*parts)]
    if op == "cost_grad":
        return {"cost": out[0], "grad": out[1]}
    if op == "refine":
        return {"center": out[0], "cost": out[1]}
    return {"center": out[0], "ok": None}


def _exact_grad(flat, w, H0, stops):
    """Score and gradient at homographies H0: eight free entries, then a marker-plane shift."""
    H = H0.clone().requires_grad_(True)
    d = torch.zeros((len(H0), 2), device=H0.device, dtype=torch.float64, requires_grad=True)
    last = H[:, :, :2] @ d[:, :, None] + H[:, :, 2:]
    G = torch.cat([H[:, :, :2], last], 2)
    p = torch.cat([stops, torch.ones_like(stops[:, :, :1])], 2)
    q = torch.einsum("nij,nkj->nki", torch.linalg.inv(G), p)
    q = q[:, :, :2] / q[:, :, 2:]
    u = _positions(H0, BEGIN[3])[None, None, :, None] * q[:, :, None, :]
    v = torch.einsum("nij,nktj->nkti", G[:, :, :2], u) + G[:, None, None, :, 2]
    cost = _score(_sample(flat, w, v[..., 0] / v[..., 2], v[..., 1] / v[..., 2]))
    gH, gd = torch.autograd.grad(cost.sum(), (H, d))
    return cost.detach(), torch.cat([gH.reshape(-1, 9)[:, :8], gd], 1)


def _exact_search(flat, w, conic, stops, c0, semi, op, steps):
    """The grid search (op "refine": its first iteration, then `steps` descent steps)."""
    semi = torch.tensor([float(np.float32(a)) for a in semi], device=c0.device, dtype=torch.float64)
    n_iter = torch.tensor([_iterations(float(a)) for a in semi], device=c0.device)
    c, ns = c0.clone(), NEIGHBOUR * semi
    offs = torch.arange(GRID, device=c0.device, dtype=torch.float64) / (GRID - 1) - 0.5
    for it in range(1 if op == "refine" else int(n_iter.max())):
        res, pts = [], []
        for i in range(GRID):
            for j in range(GRID):
                p = c + ns[:, None] * torch.stack([offs[i], offs[j]])
                pts.append(p)
                res.append(_center_score(flat, w, conic, stops, p))
        best = torch.stack(res, 1).argmin(1)
        go = (it < n_iter)[:, None]
        c = torch.where(go, torch.stack(pts, 1)[torch.arange(len(c)), best], c)
        ns = ns / 2
    if op != "refine":
        return (c,)
    alpha = 0.25 * NEIGHBOUR * semi
    best, best_cost, g = c.clone(), torch.full_like(alpha, math.inf), torch.zeros_like(c)
    for it in range(steps):
        x = c.clone().requires_grad_(True)
        cost = _center_score(flat, w, conic, stops, x)
        grad, = torch.autograd.grad(cost.sum(), x)
        better = cost.detach() < best_cost
        alpha = torch.where(better, alpha * (1.5 if it else 1.0), alpha * 0.5)
        best = torch.where(better[:, None], c, best)
        g = torch.where(better[:, None], grad, g)
        best_cost = torch.where(better, cost.detach(), best_cost)
        c = best - alpha[:, None] * g / g.norm(dim=1, keepdim=True)
    return best, best_cost
