"""Parameter gradients where the blocks of 128 Gaussians end: a full block, one more and one less, and the
half blocks past a scene's end in a batch.  Plain gradients against the FP64 reference, batched ones against
the sum of plain ones bit for bit, nothing written beyond a buffer's end.  And blends whose tiles end at a
staging round's edge: 184 splats in the backward, 256 in the forward."""
import numpy as np
import pytest

from conftest import small_scene
from test_gpu_backward import run_case
from test_gpu_batch import _plain_grads, same_bits, view_tuple

pytestmark = pytest.mark.gpu
WIDTHS = (3, 3, 4, 1, 48)


@pytest.fixture(scope="module")
def eng():
    from torpedo_amd.engine import GaussianEngine
    e = GaussianEngine()
    yield e
    e.close()


@pytest.mark.parametrize("n", [1, 127, 128, 129, 257])
def test_plain_blocks(eng, orc, n):
    run_case(eng, orc, n, 48, 40, 3, seed=n, log_scale_mean=-2.0)


@pytest.mark.parametrize("n", [183, 184, 185, 255, 256, 257, 368, 369, 553])
def test_blend_rounds(eng, orc, monkeypatch, n):
    """Faint Gaussians that all cover the one tile: every pixel blends to the end of a list of n."""
    import test_gpu_backward

    def faint(n, seed, log_scale_mean):
        g = small_scene(n, seed=seed, log_scale_mean=log_scale_mean)
        g[:, 3] = 0.012 + 0.006 * np.random.default_rng(seed).random(n, dtype=np.float32)
        return g

    monkeypatch.setattr(test_gpu_backward, "small_scene", faint)
    run_case(eng, orc, n, 16, 16, 1, seed=n, log_scale_mean=0.0)


@pytest.mark.parametrize("n", [1, 127, 128, 129, 256, 257, 385])
def test_batch_blocks(eng, n):
    from torpedo_amd.engine import GaussianEngine, Settings
    beng = GaussianEngine()
    recs = [small_scene(n, seed=n, log_scale_mean=-2.5), small_scene(n + 130, seed=n + 1, log_scale_mean=-2.5)]
    ids = [beng.addScene(r, Settings(3)) for r in recs]
    plan = [(0, (48, 33), (0.1, -0.2, -3.0)), (1, (40, 40), (0.0, 0.3, -2.8)), (0, (32, 50), (-0.6, 0.2, -2.9))]
    views = [view_tuple(ids[s], eye, w, h) for s, (w, h), eye in plan]
    beng.setViews(views)
    rng = np.random.default_rng(n)
    dls = [rng.normal(size=(h, w, 3)).astype(np.float32) for _, (w, h), _ in plan]
    dl = np.concatenate([d.reshape(-1) for d in dls])
    d_dl = beng.alloc(dl.nbytes)
    beng.upload(d_dl, dl)
    sizes = [[(r.shape[0] * k, r.shape[0] * k + 64) for k in WIDTHS] for r in recs]  # 64 floats to spare
    bufs = [[beng.alloc(4 * room) for _, room in s] for s in sizes]
    for s, bs in zip(sizes, bufs):
        for (_, room), b in zip(s, bs):
            beng.upload(b, np.full(room, 7.0, np.float32))
    beng.batchStep(d_dl, bufs)
    beng.syncBatch()
    beng.batchStep(d_dl, bufs, accumulate=True)
    beng.syncBatch()
    beng.waitIdle()
    for i, (s, bs) in enumerate(zip(sizes, bufs)):
        mine = [k for k, (sc, _, _) in enumerate(plan) if sc == i]
        ref = _plain_grads(eng, recs[i], 3, [views[k] for k in mine], [dls[k] for k in mine])
        for (used, room), b, rr, name in zip(s, bs, ref, ("means", "log_scales", "quats", "opacity_logits", "sh")):
            got = np.empty(room, np.float32)
            beng.download(got, b)
            assert np.all(got[used:] == 7.0), (i, name)
            assert same_bits(got[:used], 2.0 * rr.reshape(-1)), (i, name)  # two accumulated steps: x + x
    beng.close()
