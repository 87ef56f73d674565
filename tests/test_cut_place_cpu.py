"""The grid search reads a cut without bounds tests where cut_place has proven
its samples inside the image: the decision against the positions themselves,
on homographies whose terms cancel as far as cut_place lets them (where the
rounding of the running sums moves a sample most) and cuts that end within a
third of a pixel of the decision's 2 px margin."""
import numpy as np
import pytest

from tests import oracle_lib

INSIDE, OUTSIDE = 0, 1


def cancelling_cuts(rng, n, w, h):
    """Homographies that send t * b, t = 0.25 and 1, to two points of the image
    (near its right or left border, in its middle, just outside), the denominator's terms up to
    twenty times their sum and the numerators' up to the image's width; and the
    stops."""
    b = rng.uniform(1.7, 2.0, (n, 2)) * rng.choice([-1, 1], (n, 2))  # the longest sums of one binade
    near = rng.choice([w - 3 - 0.3, 2 + 0.3, 0.5 * w, w + 1.3], n, p=[0.7, 0.1, 0.1, 0.1])
    stop = np.stack([near + rng.uniform(-0.3, 0.3, n), rng.uniform(0.1 * h, 0.9 * h, n)], 1)
    start = stop + rng.uniform(-1, 1, (n, 2)) * [0.3, 0.05 * h]

    def row(sum_along_b, terms):
        c = terms * rng.choice([-1, 1], n)
        return np.stack([(sum_along_b / 2 + c) / b[:, 0], (sum_along_b / 2 - c) / b[:, 1]], 1)

    ratio = np.exp(rng.uniform(-0.3, 0.3, n))  # of the denominators at the two ends
    k = (ratio - 1) / (1 - 0.25 * ratio)
    H = np.ones((n, 3, 3))
    H[:, 2, :2] = row(k, np.where(rng.random(n) < 0.5, rng.uniform(0.1, 1.5, n), rng.uniform(6, 9.5, n)))
    size = np.exp(rng.uniform(np.log(0.01), np.log(0.2), n)) * w
    for a in range(2):
        n0, n1 = start[:, a] * (1 + 0.25 * k), stop[:, a] * (1 + k)
        slope = (n1 - n0) / 0.75
        H[:, a, :2], H[:, a, 2] = row(slope, size), n0 - 0.25 * slope
    return H.astype(np.float32), stop.astype(np.float32)


@pytest.mark.parametrize("w,h", [(640, 480), (1920, 1080), (7680, 4320), (32000, 16000), (60000, 8000)])
@pytest.mark.parametrize("n_samples", [31, 100, 128])
def test_decided_cuts_are_where_their_samples_are(w, h, n_samples):
    rng = np.random.default_rng(w + n_samples)
    H, stops = cancelling_cuts(rng, 400000, w, h)
    place, ext = oracle_lib.cut_places(H, stops, n_samples, w, h)
    inside = (ext[:, 0] >= 0) & (ext[:, 1] < w - 1) & (ext[:, 2] >= 0) & (ext[:, 3] < h - 1)
    assert inside[place == INSIDE].all()
    assert not inside[place == OUTSIDE].any()
    assert (place == INSIDE).mean() > 0.05 and ((place == OUTSIDE).mean() > 0.01 or w > 2**15)
    # and every cut of an ordinary marker is decided
    c, s = np.cos(0.7), np.sin(0.7)
    H = np.array([[30 * c, -30 * s, 0.4 * w], [30 * s, 30 * c, h / 2], [0.1, 0.05, 1]], np.float32)
    th = np.arange(22) * 2 * np.pi / 22
    q = H @ np.stack([np.cos(th), np.sin(th), np.ones_like(th)])
    place, _ = oracle_lib.cut_places(np.tile(H, (22, 1, 1)), (q[:2] / q[2]).T, n_samples, w, h)
    assert (place == INSIDE).all()


def test_rows_beyond_24_bit_addresses_are_not_decided_inside():
    H = np.array([[20, 0, 100], [0, 5, 12], [0, 0, 1]], np.float32)
    for w, want in ((1 << 24, 2), ((1 << 24) - 4, INSIDE)):
        place, _ = oracle_lib.cut_places(H, [[110.0, 12.0]], 100, w, 32)
        assert place[0] == want
