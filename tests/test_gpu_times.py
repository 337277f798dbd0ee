"""Stage times of profiled frames: what a frame does not run takes no time, and the parts fit the whole."""
import numpy as np
import pytest

from conftest import c1_camera, small_scene

pytestmark = pytest.mark.gpu


def test_batch_sort_times(orc):
    """The item kernel counts the pairs' digits: no histogram of theirs is timed."""
    from torpedo_amd.engine import GaussianEngine, Settings
    cam = c1_camera(orc, 320, 200)
    with GaussianEngine() as eng:
        sid = eng.addScene(small_scene(20_000, seed=1, log_scale_mean=-3.0), Settings(3))
        eng.setViews([(sid, cam.view, cam.proj_view, cam.focal_ndc, cam.width, cam.height)] * 2)
        eng.setBatchGraph(False)
        eng.setProfiling(True)
        for _ in range(2):
            eng.rasterBatch()
            eng.syncBatch()
        t, stages = eng.batchSortTimes(), eng.batchTimes()
        assert t["pair_hist_ms"] == 0.0
        assert abs(t["pair_passes_ms"] - stages["pair_sort"]) <= 1e-6
        assert abs(t["item_hist_ms"] + t["item_passes_ms"] - stages["item_sort"]) <= 1e-3
        assert t["items"] == 40_000 and t["pairs"] == eng.batchPairCount


def test_backward_times(orc):
    """Forward and backward stages lie inside the span that holds them."""
    import torch
    from torpedo_amd.engine import GaussianEngine
    n, cam = 50_000, c1_camera(orc, 320, 200)
    with GaussianEngine() as eng:
        eng.uploadRecords(small_scene(n, seed=2, log_scale_mean=-3.0), 3)
        eng.setCamera(cam.view, cam.proj_view, cam.focal_ndc, cam.width, cam.height)
        up = torch.ones(200, 320, 3, device="cuda")
        out = [torch.empty(n, k, device="cuda") for k in (3, 3, 4, 1, 48)]
        torch.cuda.synchronize()
        eng.setProfiling(True)
        for _ in range(2):
            eng.render()
            eng.backward(up.data_ptr(), *[t.data_ptr() for t in out])
        fwd, bwd = eng.stageTimes(), eng.backwardTimes()
        assert min(bwd.values()) > 0.0 and np.isfinite(list(bwd.values())).all()
        assert fwd["frame"] + bwd["splat_grad_pass"] + bwd["param_grad_pass"] <= bwd["fwd_bwd_span"] + 1e-3


def test_stage_times_of_a_frame_without_room(orc):
    """A first frame of more pairs than there is room for emits them twice and grows its buffers between:
    that is in no stage's time, only in the whole frame's."""
    from torpedo_amd.engine import GaussianEngine
    cam = c1_camera(orc, 320, 200)
    with GaussianEngine() as eng:
        eng.uploadRecords(small_scene(200_000, seed=3, log_scale_mean=-0.5), 3)
        eng.setCamera(cam.view, cam.proj_view, cam.focal_ndc, cam.width, cam.height)
        eng.setProfiling(True)
        eng.render()
        first = eng.stageTimes()
        assert eng.frameIssues() == (1, 1) and eng.pairCount > 5 * 200_000
        for _ in range(3):
            eng.render()
        then = eng.stageTimes()
        assert eng.frameIssues() == (4, 1)
        stages = [k for k in first if k not in ("frame", "radix_passes")]
        gap = first["frame"] - sum(first[k] for k in stages)
        assert gap > then["frame"] - sum(then[k] for k in stages)
        # the item passes wait for nothing
        assert first["sort_passes"] <= 2.0 * then["sort_passes"] + 0.2, (first, then)
