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
    """One frame, checked; returns how often it was issued, and its pairs issued again."""
    before = eng.frameIssues()
    eng.setCamera(cam.view, cam.proj_view, cam.focal_ndc, cam.width, cam.height)
    eng.render()
    keys, vals = eng.readPairs()
    ref = orc.render(g, cam, 3)
    assert np.array_equal(keys, ref["keys"]) and np.array_equal(vals, ref["vals"])
    assert np.abs(eng.readImage() - ref["image"]).max() <= 1e-5
    return tuple(a - b for a, b in zip(eng.frameIssues(), before))


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
    assert frame(eng, orc, g, inside) == (1, 0) and eng.stageTimes()["radix_passes"] == 4
    assert frame(eng, orc, g, outside) == (2, 0) and eng.stageTimes()["radix_passes"] == 5
    for k in range(12):
        assert frame(eng, orc, g, (inside, outside)[k % 2]) == (1, 0), k
    for k in range(64):
        assert frame(eng, orc, g, inside) == (1, 0) and eng.stageTimes()["radix_passes"] == 5, k
    assert frame(eng, orc, g, inside) == (1, 0) and eng.stageTimes()["radix_passes"] == 4
    assert frame(eng, orc, g, outside) == (2, 0)


def crowd(n, seed, scale, far=None):
    """n Gaussians of n x some hundred pairs at 320x200; far: and one at that depth."""
    g = small_scene(n, seed=seed, log_scale_mean=scale)
    if far is not None:
        from torpedo_amd.engine import gaussian_point
        g = np.concatenate([g, gaussian_point([0, 0, far], 0.8, (0, 0, 0, 1), (2.0,) * 3, np.full(48, 0.3, np.float32))[None]])
    return g


@pytest.mark.parametrize("shape", [None, 0, 6, 9])
def test_first_frame_over_the_room(orc, shape):
    """More pairs than max(4 n, 2^20) with headroom: the Gaussians are projected and sorted once, their pairs
    emitted again with room for them; then the same frame, a backward and a small frame."""
    from torpedo_amd.engine import GaussianEngine
    cam = orc.make_camera([0.0, 0.0, -3.0], [0.0, 0.0, 0.0], [0.0, -1.0, 0.0], W, H)
    g, small = crowd(8000, 11, -0.5), crowd(500, 12, -3.0)
    with GaussianEngine() as eng:
        if shape is not None:
            eng.setSortShape(shape)
        eng.uploadRecords(g, 3)
        assert frame(eng, orc, g, cam) == (1, 1) and eng.pairCount > 5 * (1 << 18)
        assert frame(eng, orc, g, cam) == (1, 0)
        counts, offs = eng.readTiles()
        assert counts.sum() == eng.pairCount and np.array_equal(offs[1:], np.cumsum(counts)[:-1])
        eng.uploadRecords(small, 3)
        assert frame(eng, orc, small, cam) == (1, 0)


def test_first_frame_over_the_room_and_the_window(orc, eng):
    """A first frame with neither room for its pairs nor its depths in the window."""
    cam = orc.make_camera([0.0, 0.0, -3.0], [0.0, 0.0, 0.0], [0.0, -1.0, 0.0], W, H, near=0.01, far=1000.0)
    g = crowd(8000, 13, -0.5, far=300.0)
    eng.uploadRecords(g, 3)
    assert frame(eng, orc, g, cam) == (2, 0) and eng.pairCount > 5 * (1 << 18)
    assert frame(eng, orc, g, cam) == (1, 0)


def test_backward_of_a_resumed_frame(orc):
    """The gradients of a frame whose pairs were emitted twice are those of the frame issued with room."""
    import torch
    from torpedo_amd.engine import GaussianEngine
    cam = orc.make_camera([0.0, 0.0, -3.0], [0.0, 0.0, 0.0], [0.0, -1.0, 0.0], W, H)
    g = crowd(8000, 14, -0.5)
    with GaussianEngine() as eng:
        up = torch.randn(H, W, 3, device="cuda", generator=torch.Generator("cuda").manual_seed(3))
        sets = [[torch.empty(g.shape[0], k, device="cuda") for k in (3, 3, 4, 1, 48)] for _ in range(2)]
        torch.cuda.synchronize()
        eng.uploadRecords(g, 3)
        for k, out in enumerate(sets):
            assert frame(eng, orc, g, cam) == (1, 1 - k)
            eng.backward(up.data_ptr(), *[t.data_ptr() for t in out])
            eng.waitIdle()
        assert all(torch.equal(a, b) for a, b in zip(*sets))


def test_room_follows_recent_frames(orc, eng):
    """A large frame by turns with small ones keeps its room; forty small frames later it has to find it
    again (and small frames no longer run over it)."""
    cam = orc.make_camera([0.0, 0.0, -3.0], [0.0, 0.0, 0.0], [0.0, -1.0, 0.0], W, H)
    large, small = crowd(8000, 15, -0.5), crowd(500, 16, -3.0)

    def show(g):
        eng.uploadRecords(g, 3)
        return frame(eng, orc, g, cam)

    assert show(large) == (1, 1) and show(large) == (1, 0)
    for _ in range(3):
        assert show(small) == (1, 0) and show(large) == (1, 0)
    eng.uploadRecords(small, 3)
    for _ in range(40):
        assert frame(eng, orc, small, cam) == (1, 0)
    assert show(large) == (1, 1) and show(large) == (1, 0) and show(small) == (1, 0)


def test_room_of_the_widest_view(orc, eng):
    """One view in thirty with three times the others' pairs: it finds its room each time."""
    g = crowd(8000, 15, -0.5)
    near, far = (orc.make_camera([0.0, 0.0, z], [0.0, 0.0, 0.0], [0.0, -1.0, 0.0], W, H) for z in (-3.0, -40.0))
    eng.uploadRecords(g, 3)
    assert frame(eng, orc, g, near) == (1, 1)
    pairs = eng.pairCount
    for _ in range(3):
        for k in range(29):
            eng.setCamera(far.view, far.proj_view, far.focal_ndc, far.width, far.height)
            eng.render()
        assert 3 * eng.pairCount < pairs
        assert frame(eng, orc, g, near) == (1, 0)


@pytest.mark.parametrize("n,scale", [(8_000, -0.5), (40_000, -0.5), (9_000, -1.7)])
def test_first_batch_over_the_room(orc, n, scale):
    """A batch's first frame with many times the pairs its buffers hold, blocks of it all past their end:
    each view's pairs and image are the plain frame's."""
    from torpedo_amd.engine import GaussianEngine, Settings
    g = small_scene(n, seed=n, log_scale_mean=scale)
    cams = [orc.make_camera([x, 0.0, -3.0], [0.0, 0.0, 0.0], [0.0, -1.0, 0.0], W, H) for x in (0.0, 0.4)]
    with GaussianEngine() as eng, GaussianEngine() as plain:
        sid = eng.addScene(g, Settings(3))
        eng.setViews([(sid, c.view, c.proj_view, c.focal_ndc, c.width, c.height) for c in cams])
        eng.rasterBatch()
        keys, vals = eng.readBatchPairs()
        plain.uploadRecords(g, 3)
        for v, c in enumerate(cams):
            plain.setCamera(c.view, c.proj_view, c.focal_ndc, c.width, c.height)
            plain.render()
            tile0, item0, _ = eng.batchViewLayout(v)
            pk, pv = plain.readPairs()
            mine = (vals >= item0) & (vals < item0 + n)
            assert np.array_equal(vals[mine] - item0, pv)
            assert np.array_equal(keys[mine] - (np.uint64(tile0) << np.uint64(32)), pk)
            assert np.array_equal(eng.readBatchImage(v), plain.readImage())
