"""A frame issued behind long work on its stream: the caller's thread sleeps while it waits."""
import time

import numpy as np
import pytest

from conftest import c1_camera, small_scene

pytestmark = pytest.mark.gpu


def test_frame_behind_long_work(orc):
    import torch
    from torpedo_amd.engine import GaussianEngine
    n, cam = 3_000, c1_camera(orc, 160, 96)
    g = small_scene(n, seed=4, log_scale_mean=-3.0)
    x = torch.ones(8192, 8192, device="cuda", dtype=torch.bfloat16)
    y, side = torch.empty_like(x), torch.cuda.Stream()
    torch.mm(x, x, out=y)
    torch.cuda.synchronize()
    with GaussianEngine() as eng:
        eng.uploadRecords(g, 3)
        eng.setCamera(cam.view, cam.proj_view, cam.focal_ndc, cam.width, cam.height)
        eng.render(side.cuda_stream)
        side.synchronize()
        with torch.cuda.stream(side):
            for _ in range(100):  # at least 44 ms: 110 TFLOP at 2.5 PFLOP/s
                torch.mm(x, x, out=y)
        wall, cpu = time.perf_counter(), time.thread_time()
        eng.render(side.cuda_stream)
        wall, cpu = time.perf_counter() - wall, time.thread_time() - cpu
        side.synchronize()
        assert np.abs(eng.readImage() - orc.render(g, cam, 3)["image"]).max() <= 1e-5
    # what was not awake: all but the first 10 ms, the launches and the looks
    assert wall >= 0.03 and cpu <= 0.5 * wall, (wall, cpu)
