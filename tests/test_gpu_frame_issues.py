"""How often a plain frame is issued, and with what: sequences whose depths move in and out of the sort's
depth window, frames with more pairs than there is room for, and small frames after large ones.  Every
frame is compared with the oracle too."""
import numpy as np
import pytest

from conftest import small_scene

pytestmark = pytest.mark.gpu
W, H = 320, 200


@pytest.fixture()
def eng():
    from torpedo_amd.engine import GaussianEngine
    e = GaussianEngine()
    yield e
    e.close()


def frame(eng, orc, g, cam):
    """One frame, checked; returns how often it was issued."""
    before = eng.frameIssues()
    eng.setCamera(cam.view, cam.proj_view, cam.focal_ndc, cam.width, cam.height)
    eng.render()
    keys, vals = eng.readPairs()
    ref = orc.render(g, cam, 3)
    assert np.array_equal(keys, ref["keys"]) and np.array_equal(vals, ref["vals"])
    assert np.abs(eng.readImage() - ref["image"]).max() <= 1e-5
    return eng.frameIssues() - before


def test_depths_moving_across_the_window(eng, orc):
    """One Gaussian's depth is 255 or 257 by turns: the wide key is found once and kept.  It is given up
    after 64 frames without such a depth (a 9-bit shape: 9 + 27 bits in 4 passes, 9 + 31 in 5)."""
    from torpedo_amd.engine import gaussian_point
    far = gaussian_point([0, 0, 254.0], 0.8, (0, 0, 0, 1), (2.0,) * 3, np.full(48, 0.3, np.float32))[None]
    g = np.concatenate([small_scene(3000, seed=3, log_scale_mean=-3.0), far])
    inside, outside = (orc.make_camera([0.0, 0.0, z], [0.0, 0.0, 10.0], [0.0, -1.0, 0.0], W, H, near=0.01, far=1000.0)
                       for z in (-1.0, -3.0))
    for cam, at in ((inside, 255.0), (outside, 257.0)):
        sp = orc.render(g, cam, 3)["splats"]
        assert sp["tiles"][-1] > 0 and sp["texel"][-1, 2] == np.float32(at)
    eng.uploadRecords(g, 3)
    eng.setSortShape(6)
    eng.setProfiling(True)
    assert frame(eng, orc, g, inside) == 1 and eng.stageTimes()["radix_passes"] == 4
    assert frame(eng, orc, g, outside) == 2 and eng.stageTimes()["radix_passes"] == 5
    for k in range(12):
        assert frame(eng, orc, g, (inside, outside)[k % 2]) == 1, k
    for k in range(64):
        assert frame(eng, orc, g, inside) == 1 and eng.stageTimes()["radix_passes"] == 5, k
    assert frame(eng, orc, g, inside) == 1 and eng.stageTimes()["radix_passes"] == 4
    assert frame(eng, orc, g, outside) == 2
