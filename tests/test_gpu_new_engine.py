"""An engine's first frames, plain and batched, while another thread keeps the device's null stream busy:
what the engine clears on that stream when it allocates must be clear before frames on other streams use it."""
import threading

import numpy as np
import pytest

from conftest import c1_camera, small_scene

pytestmark = pytest.mark.gpu


def test_first_frames_beside_a_busy_null_stream(orc):
    import torch
    from torpedo_amd.engine import GaussianEngine, Settings
    n, cam = 3_000, c1_camera(orc, 160, 96)
    g = small_scene(n, seed=9, log_scale_mean=-3.0)
    want = orc.render(g, cam, 3)["image"]
    stop = threading.Event()

    def busy():  # a few milliseconds of queued products at a time, never more
        x = torch.randn(4096, 4096, device="cuda")
        y = torch.empty_like(x)
        while not stop.is_set():
            for _ in range(8):
                torch.mm(x, x, out=y)
            torch.cuda.default_stream().synchronize()

    t = threading.Thread(target=busy)
    t.start()
    try:
        for _ in range(20):
            with GaussianEngine() as eng:
                eng.uploadRecords(g, 3)
                eng.setCamera(cam.view, cam.proj_view, cam.focal_ndc, cam.width, cam.height)
                eng.render()
                assert np.abs(eng.readImage() - want).max() <= 1e-5
                view = (eng.addScene(g, Settings(3)), cam.view, cam.proj_view, cam.focal_ndc, cam.width, cam.height)
                eng.setViews([view, view])
                eng.rasterBatch()
                assert all(np.abs(eng.readBatchImage(v) - want).max() <= 1e-5 for v in (0, 1))
    finally:
        stop.set()
        t.join()
