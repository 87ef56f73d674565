"""How the score's float sampling rounds.  A homography and its multiples are
one map.  With samples on positions that a float holds exactly, and quotients
and the adjoint's 1 / w correctly rounded or in double, a multiple's samples
are the same: the score is equal and the gradient is the first one over the
factor, to double rounding.  A rounded float reciprocal in either place would
show at 1e-8 to 1e-7, on pixel borders (where many of these samples lie) at
any size."""
import numpy as np
import pytest

from cctag_amd import _lib
from cctag_amd.detector import Refiner

# 97 samples from 0.25 to 1: steps of 2^-7
N_SAMPLES = 97
STOPS = [[80, 70], [50, 60], [66, 90], [71, 40], [58, 50], [75, 75], [40, 81], [90, 61], [64, 88]]


@pytest.mark.gpu
@pytest.mark.parametrize("factor", [3, 5, 7, 11, -13, 2.0**70, -2.0**-70])  # (the last two: w out of div2_rn's range)
@pytest.mark.parametrize("shift", [0, 1792])
def test_multiples_of_a_homography(factor, shift):
    y, x = np.mgrid[0:128, 0:128 + shift]
    img = (127 + 60 * np.sin(x / 5.0) + 60 * np.cos(y / 7.0)).astype(np.uint8)
    H = np.array([[[16, 0, 64 + shift], [0, 16, 64], [0, 0, 1]]], np.float32)
    p = _lib.default_params(3)
    p.sample_cut_length = N_SAMPLES
    stops = np.array(STOPS, float) + [shift, 0]
    with Refiner(1, p) as r:
        r.set_image(img)
        r.set_markers([{"ellipse": (64.0 + shift, 64.0, 16.0, 16.0, 0.0),
                        "center0": (64.0 + shift, 64.0), "stops": stops}])
        c1, g1 = r.cost_grad(H)
        cf, gf = r.cost_grad(np.float32(factor) * H)
    gf[0, :8] *= factor
    print(factor, shift, c1, cf, flush=True)
    # double rounding: sums of fewer than 1000 terms in 2^-53
    assert abs(cf[0] - c1[0]) <= 1e-12 * c1[0]
    assert np.linalg.norm(gf - g1) <= 1e-12 * np.linalg.norm(g1)
