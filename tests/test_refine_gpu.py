"""The grid search's two kernels (one launch per iteration for few markers, a
block per marker for many) at the edges of their shapes: every split of the
samples over blocks, partial chunks, the fewest and most cuts,
markers cut by the image border.  A marker's result must not depend,
bit for bit, on how many others are searched with it; interior markers are
checked against the same search in float64."""
import numpy as np
import pytest

from cctag_amd import _lib, synth
from cctag_amd.detector import Refiner

FIRST_BLOCK_PER_MARKER = 150  # markers from which the second kernel runs


def grid(img, markers, params):
    with Refiner(len(markers), params) as r:
        r.set_image(img)
        r.set_markers(markers)
        c, ok = r.grid()
    return c.view(np.int32), ok


def grid64(img, m, n_samples, grid_n=5, begin=0.25, neighbour=0.2):
    """The search of one marker whose cuts all stay inside the image, in
    float64: the polar of the centre is the marker plane's vanishing line,
    which weighs the projective segment from the centre to a stop."""
    im = img.astype(np.float64)
    cx, cy, a, b, ang = m["ellipse"]
    c, s = np.cos(ang), np.sin(ang)
    M = np.array([[c / a, s / a, -(c * cx + s * cy) / a], [-s / b, c / b, (s * cx - c * cy) / b],
                  [0, 0, 1.0]])
    conic = M.T @ np.diag([1.0, 1.0, -1.0]) @ M
    t = begin + np.arange(n_samples) * (1 - begin) / (n_samples - 1)
    stops = np.asarray(m["stops"], np.float32).astype(np.float64)

    def score(p):
        line = conic @ np.array([p[0], p[1], 1.0])
        wc = 1 / (line[:2] @ p + line[2])
        wp = 1 / (stops @ line[:2] + line[2])
        u, v = t * wp[:, None], (1 - t) * wc
        x = (u * stops[:, :1] + v * p[0]) / (u + v)
        y = (u * stops[:, 1:] + v * p[1]) / (u + v)
        ix, iy = x.astype(int), y.astype(int)
        fx, fy = x - ix, y - iy
        val = ((im[iy, ix] * (1 - fx) + im[iy, ix + 1] * fx) * (1 - fy) +
               (im[iy + 1, ix] * (1 - fx) + im[iy + 1, ix + 1] * fx) * fy)
        k = len(stops)
        return (k * (val ** 2).sum(0) - val.sum(0) ** 2).sum()

    p, size = np.array(m["center0"], np.float64), neighbour * max(a, b)
    offs = np.arange(grid_n) / (grid_n - 1) - 0.5
    while size > 0.02:
        pts = [p + size * np.array([i, j]) for i in offs for j in offs]
        p = pts[int(np.argmin([score(q) for q in pts]))]
        size /= (grid_n - 1) // 2
    return p


def params(n_samples=100):
    p = _lib.default_params(3)
    p.sample_cut_length = n_samples
    return p


@pytest.mark.gpu
@pytest.mark.parametrize("n_samples,n_cuts", [(100, 22), (31, 2), (128, 32), (45, 32), (100, 7)])
def test_both_kernels_agree_and_match_float64(n_samples, n_cuts):
    img, ms = synth.refine_mosaic(16, unique=16, seed=77)
    rng = np.random.default_rng(n_samples)
    for m in ms:  # the cuts asked for, spread over the outer ellipse
        H = m["H"]
        th = rng.uniform(0, 1) + 2 * np.pi * np.arange(n_cuts) / n_cuts
        q = H @ np.stack([np.cos(th), np.sin(th), np.ones_like(th)])
        m["stops"] = (q[:2] / q[2]).T
    p = params(n_samples)
    few, ok_few = grid(img, ms, p)
    assert ok_few.all()
    many, ok_many = grid(img, ms * 10, p)  # 160 markers
    assert len(ms) * 10 >= FIRST_BLOCK_PER_MARKER
    assert ok_many.all() and np.array_equal(many, np.tile(few, (10, 1)))
    # 112 and 52 markers: several chunks per block, so two sample buffers (with
    # 32 cuts the most LDS a block takes) and blocks that end on a partial chunk
    for n in (112, 52):
        got, ok = grid(img, (ms * 7)[:n], p)
        print("split over blocks", n_samples, n_cuts, n, flush=True)
        assert ok.all() and np.array_equal(got, np.tile(few, (7, 1))[:n])
    if n_cuts >= 7:  # (two cuts leave the minimum undetermined along a line)
        # the centres of two equal searches agree within the pixel tolerance
        # that the detection tests hold (float sampling moves a near tie)
        want = np.array([grid64(img, m, n_samples) for m in ms[:6]])
        assert np.abs(few.view(np.float32)[:6] - want).max() < 0.05


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 51, 52, 103, 149, 150, 257])
def test_a_marker_does_not_depend_on_the_others(n):
    img, gts = synth.border_frame()
    ms = [synth.refine_marker(g.H) for g in gts]  # four of them cut by the border
    few, few_ok = grid(img, ms, params())  # (the first marker conditions all of them)
    got, ok = grid(img, [ms[i % len(ms)] for i in range(n)], params())
    for i in range(n):
        j = i % len(ms)
        assert ok[i] == few_ok[j] and np.array_equal(got[i], few[j]), (n, i)
