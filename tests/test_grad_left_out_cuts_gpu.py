"""A cut that cannot be sampled -- its stop is not finite, or lies on the
marker plane's vanishing line -- is left out of the score, of its gradient and
of the descent: the results are those of the marker without that cut."""
import numpy as np
import pytest

from cctag_amd import synth
from cctag_amd.detector import Refiner
from tests import oracle_lib

NAN, INF = float("nan"), float("inf")


def plane(w=192, h=128):
    y, x = np.mgrid[0:h, 0:w]
    return (127 + 60 * np.sin(x / 5.0) + 60 * np.cos(y / 7.0)).astype(np.uint8)


def marker(stops):
    return {"ellipse": (96.0, 64.0, 20.0, 16.0, 0.0), "center0": (96.0, 64.0), "stops": np.array(stops)}


# exact in float: the centre is (96, 64) and the image of the plane's points
# at infinity x = 64
HOM = np.array([[[16, 0, 96], [0, 16, 64], [0.25, 0, 1]]], np.float32)
GOOD = [[80.0, 70.0], [110.0, 60.0], [96.5, 90.0], [101.0, 40.0], [88.0, 50.0], [105.0, 75.0]]


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [[64.0, 80.0], [NAN, 60.0], [INF, INF]], ids=["vanishing", "nan", "inf"])
@pytest.mark.parametrize("at", [0, 3, 6])
def test_score_and_gradient_without_the_cut(bad, at):
    img = plane()
    stops = GOOD[:at] + [bad] + GOOD[at:]
    got = []
    for s in (GOOD, stops):
        with Refiner(1) as r:
            r.set_image(img)
            r.set_markers([marker(s)])
            got.append([r.cost_grad(HOM), r.cost_grad(HOM, fp64=True)])
    c, _, nv = oracle_lib.grad_cost(img, HOM[0].astype(np.float64), GOOD, grad=False)
    assert nv == len(GOOD)
    assert abs(got[1][1][0][0] - c) <= 1e-9 * c
    # (the gradient is compared with the kernel's own only: stops on whole pixels
    # are kinks of the bilinear image, where the oracle may take the other side)
    for (c0, g0), (c1, g1) in zip(*got):  # the cuts' terms may add up in another order
        assert np.isfinite(g1).all() and abs(c1 - c0) <= 1e-12 * c0
        assert np.linalg.norm(g1 - g0) <= 1e-12 * np.linalg.norm(g0)


@pytest.mark.gpu
@pytest.mark.parametrize("fp64", [False, True])
def test_descent_without_the_cut(fp64):
    img, ms = synth.refine_mosaic(4, unique=4, seed=21)
    out = []
    for extra in ([], [[NAN, 10.0]]):
        with Refiner(len(ms)) as r:
            r.set_image(img)
            r.set_markers([dict(m, stops=np.array(list(m["stops"]) + extra)) for m in ms])
            out.append([*r.descend(12, fp64=fp64), *r.refine(12, fp64=fp64)])
    assert np.abs(out[0][0] - [m["center0"] for m in ms]).max() > 0.05  # it moved
    for a, b in zip(*out):
        assert a.tobytes() == b.tobytes()
