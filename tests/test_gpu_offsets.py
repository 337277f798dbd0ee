"""Pair offsets of a plain frame wherever they are asked for: read back while the frame still runs on a
caller's stream, after backwards on it, in a second backward of one frame, and in a backward that was
recorded into a graph and is replayed for later frames."""
import numpy as np
import pytest

from conftest import c1_camera, small_scene

pytestmark = pytest.mark.gpu
WIDTHS = (3, 3, 4, 1, 48)
W, H = 320, 208


def set_camera(eng, cam):
    eng.setCamera(cam.view, cam.proj_view, cam.focal_ndc, cam.width, cam.height)


def device_scene(eng, g):
    import torch
    rec = torch.from_numpy(np.ascontiguousarray(g)).cuda()
    torch.cuda.synchronize()
    eng.bindDeviceScene(rec.data_ptr(), g.shape[0], 3)
    return rec


def backward(eng, up, out, stream=None):
    eng.backward(up.data_ptr(), *[t.data_ptr() for t in out], stream=stream)


@pytest.mark.parametrize("n", [700, 40_000])
@pytest.mark.parametrize("backwards", [0, 1, 2])
def test_tiles_read_after_other_streams(orc, n, backwards):
    """A training loop's frame and backwards on a stream of the caller's, then another scene's frame there:
    its tiles are read at once, by the engine's own stream."""
    import torch
    from torpedo_amd.engine import GaussianEngine
    cam = c1_camera(orc, W, H)
    scenes = [small_scene(n, seed=s, log_scale_mean=m) for s, m in ((1, -2.5), (2, -3.5), (3, -2.8))]
    s = torch.cuda.Stream()
    with GaussianEngine() as eng:
        up = torch.ones(H, W, 3, device="cuda")
        out = [torch.empty(n, k, device="cuda") for k in WIDTHS]
        for g in scenes:
            rec = device_scene(eng, g)
            set_camera(eng, cam)
            eng.render(s.cuda_stream)
            counts, offs = eng.readTiles()
            ref = orc.preprocess(g, cam, 3)["tiles"]
            assert np.array_equal(counts, ref)
            assert np.array_equal(offs, np.concatenate([[0], np.cumsum(ref, dtype=np.uint64)[:-1]]).astype(np.uint32))
            for _ in range(backwards):
                backward(eng, up, out, s.cuda_stream)
            s.synchronize()
            del rec


def test_second_backward_of_a_frame(orc):
    """Two backwards of one frame, a readback between them: the same bits, and twice them when added."""
    import torch
    from torpedo_amd.engine import GaussianEngine
    n, cam = 5_000, c1_camera(orc, W, H)
    with GaussianEngine() as eng:
        rec = device_scene(eng, small_scene(n, seed=4, log_scale_mean=-3.0))
        set_camera(eng, cam)
        eng.render()
        up = torch.randn(H, W, 3, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
        torch.cuda.synchronize()
        first, second = ([torch.empty(n, k, device="cuda") for k in WIDTHS] for _ in range(2))
        backward(eng, up, first)
        eng.readTiles()
        backward(eng, up, second)
        eng.waitIdle()
        assert all(torch.equal(a, b) for a, b in zip(first, second))
        assert all(bool((t != 0).any()) for t in first)
        del rec


def test_recorded_backward(orc):
    """A backward recorded into a graph after an eager one, replayed for frames whose records and transform
    have changed since: each replay against the eager backward of its frame."""
    import torch
    from torpedo_amd.engine import Entity, GaussianEngine
    n, cam = 3_000, c1_camera(orc, W, H)
    with GaussianEngine() as eng:
        # the first scene has the most pairs: the buffer of partial sums is sized by its frame
        recs = [torch.from_numpy(small_scene(n, seed=s, log_scale_mean=m)).cuda() for s, m in
                ((5, -2.4), (6, -3.0), (7, -3.4), (8, -2.8))]
        rec = recs[0].clone()
        up = torch.randn(H, W, 3, device="cuda", generator=torch.Generator("cuda").manual_seed(2))
        grads = [torch.empty(n, k, device="cuda") for k in WIDTHS]
        torch.cuda.synchronize()
        eng.bindDeviceScene(rec.data_ptr(), n, 3)
        set_camera(eng, cam)
        s = torch.cuda.Stream()
        eng.render(s.cuda_stream)
        backward(eng, up, grads, s.cuda_stream)
        s.synchronize()
        most = eng.pairCount
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            backward(eng, up, grads, s.cuda_stream)
        shift = np.eye(4, dtype=np.float32)
        for k, r in enumerate(recs + recs):
            rec.copy_(r)
            torch.cuda.synchronize()
            shift[0, 3] = 0.05 * k
            eng.getTransformHost().transform(Entity(0), shift)
            eng.render(s.cuda_stream)
            assert eng.pairCount <= most * 5 // 4  # the room the partial sums were given
            s.synchronize()
            for t in grads:
                t.fill_(7.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            replayed = [t.clone() for t in grads]
            torch.cuda.synchronize()
            backward(eng, up, grads, s.cuda_stream)
            s.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(replayed, grads)), k
