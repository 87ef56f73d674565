"""A refiner's markers after a set that was refused: the set before it stays
in force, whole, for every call that uses it."""
import numpy as np
import pytest

from cctag_amd import synth
from cctag_amd.detector import Refiner


def results(r, H):
    return [np.ascontiguousarray(a).tobytes()
            for a in (*r.cost_grad(H), *r.cost_grad(H, fp64=True), r.homography(H[:, :2, 2]),
                      *r.descend(5), *r.refine(5), *r.grid())]


@pytest.mark.gpu
@pytest.mark.parametrize("refused", ["cuts", "ellipse", "shorter", "longer"])
def test_a_refused_marker_set_leaves_the_one_before(refused):
    img, gts = synth.border_frame()
    ms = [synth.refine_marker(g.H, 22) for g in gts[:4]]
    H = np.array([m["H"] / m["H"][2, 2] for m in ms], np.float32)
    one_cut = dict(ms[0], stops=ms[0]["stops"][:1])
    few = dict(ms[1], stops=ms[1]["stops"][:2])
    flat = dict(few, ellipse=(60.0, 60.0, -1.0, 20.0, 0.0))
    bad = {"cuts": [one_cut, few, few, few], "ellipse": [few, few, few, flat],
           "shorter": [few, one_cut], "longer": [few] * 6 + [one_cut]}[refused]
    with Refiner(8) as r:
        r.set_image(img)
        r.set_markers(ms)
        want = results(r, H)
        with pytest.raises(RuntimeError):
            r.set_markers(bad)
        print("refused", refused, flush=True)
        assert results(r, H) == want
        r.set_markers([few, few])
        assert len(r.grid()[1]) == 2
