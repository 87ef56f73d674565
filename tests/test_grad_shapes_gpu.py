"""The differentiable score's kernels at the edges of their shapes (fewest and
most cuts, every count of samples a lane keeps, cuts outside the image)
against the float64 oracle."""
import numpy as np
import pytest

from cctag_amd import _lib, synth
from cctag_amd.detector import Refiner
from tests import oracle_lib


def stops_on(H, n_cuts, phase):
    th = phase + 2 * np.pi * np.arange(n_cuts) / n_cuts
    q = H @ np.stack([np.cos(th), np.sin(th), np.ones_like(th)])
    return (q[:2] / q[2]).T


@pytest.mark.gpu
@pytest.mark.parametrize("n_samples,n_cuts", [(100, 22), (31, 2), (104, 32), (105, 32), (128, 9)])
def test_score_and_gradient_shapes(n_samples, n_cuts):
    img, gts = synth.border_frame()  # four markers cut by the border, two whole
    ms = [synth.refine_marker(g.H) for g in gts]
    for i, m in enumerate(ms):
        m["stops"] = stops_on(m["H"], n_cuts, 0.3 + i)
    p = _lib.default_params(3)
    p.sample_cut_length = n_samples
    H = np.array([m["H"] @ np.array([[1, 0, 0.01], [0, 1, -0.02], [0, 0, 1.0]]) for m in ms])
    H = (H / H[:, 2:, 2:]).astype(np.float32)
    with Refiner(len(ms), p) as r:
        r.set_image(img)
        r.set_markers(ms)
        cost64, grad64 = r.cost_grad(H, fp64=True)
        cost32, grad32 = r.cost_grad(H)
    scored = 0
    for i, m in enumerate(ms):
        c, g, nv = oracle_lib.grad_cost(img, H[i].astype(np.float64), m["stops"], n_samples)
        if nv < 2:
            assert cost64[i] == cost32[i] == np.finfo(np.float64).max
            assert not grad64[i].any() and not grad32[i].any()
            continue
        scored += 1
        # the bounds of the default shape's test: fp64 sampling to 1e-9 / 1e-7,
        # float sampling to 2e-3 / 1e-2
        g8 = np.ravel(g)[:8]
        assert abs(cost64[i] - c) <= 1e-9 * c
        assert np.linalg.norm(grad64[i, :8] - g8) <= 1e-7 * np.linalg.norm(g8)
        assert abs(cost32[i] - c) <= 2e-3 * c
        assert np.linalg.norm(grad32[i] - grad64[i]) <= 1e-2 * np.linalg.norm(grad64[i])
    assert scored >= 2
