"""Which launch shape the sorts run with: a frame's autotune leaves the stand-alone sorts' alone, and a
selected or tuned shape can be given back.  The number of passes tells the digit width: an odd one leaves the
result in the other buffers."""
import ctypes

import numpy as np
import pytest

from conftest import c1_camera, small_scene

pytestmark = pytest.mark.gpu
BITS = (17, 43, 45, 54, 63)  # widths whose 8- and 9-bit digits need an odd and an even number of passes


def sort_in_alt(eng, bits, noalloc=False, n=5_000):
    """Sorts n keys of so many bits, checks the result, and tells where it was left."""
    import torch
    from torpedo_amd.engine import sort_pairs_device, sort_pairs_device_noalloc
    keys = np.random.default_rng(bits).integers(0, 2 ** bits, n, dtype=np.uint64)
    k = torch.from_numpy(keys.view(np.int64)).cuda()
    v = torch.arange(n, dtype=torch.int32, device="cuda")
    ka, va = torch.empty_like(k), torch.empty_like(v)
    torch.cuda.synchronize()
    sort = sort_pairs_device_noalloc if noalloc else sort_pairs_device
    alt = sort(eng, k.data_ptr(), v.data_ptr(), ka.data_ptr(), va.data_ptr(), n, bits)
    eng.waitIdle()
    assert np.array_equal((va if alt else v).cpu().numpy(), np.argsort(keys, kind="stable"))
    return alt


@pytest.mark.parametrize("n,w,h", [(3_000, 64, 64), (100_000, 1280, 720)])
def test_autotune_leaves_the_stand_alone_sorts(orc, n, w, h):
    from torpedo_amd.engine import GaussianEngine
    with GaussianEngine() as eng:
        eng.uploadRecords(small_scene(n, seed=n, log_scale_mean=-3.5), 3)
        cam = c1_camera(orc, w, h)
        eng.setCamera(cam.view, cam.proj_view, cam.focal_ndc, cam.width, cam.height)
        eng.render()
        before = [sort_in_alt(eng, b, na) for b in BITS for na in (False, True)]
        assert before == [((b + 8) // 9) % 2 == 1 for b in BITS for _ in (0, 1)]  # 9-bit digits save a pass
        image = eng.readImage()
        eng.autotune()
        assert [sort_in_alt(eng, b, na) for b in BITS for na in (False, True)] == before
        assert np.array_equal(eng.readImage(), image)


def batch_shapes(eng):
    from torpedo_amd._capi import check, lib
    item, pair = ctypes.c_uint32(), ctypes.c_uint32()
    check(lib().tpd_batch_get_sort_shapes(eng._ctx, ctypes.byref(item), ctypes.byref(pair)))
    return item.value, pair.value


def test_a_shape_given_back(orc):
    """A selected shape, then an autotune of the frame and one of the batch: after each, all sorts run again
    with the shapes of an engine that never had another, and the frames are the same bits."""
    from torpedo_amd.engine import GaussianEngine, Settings
    g, cam = small_scene(60_000, seed=8, log_scale_mean=-3.5), c1_camera(orc, 640, 360)

    def shapes(eng):
        eng.render()
        eng.rasterBatch()
        eng.syncBatch()
        return ([sort_in_alt(eng, b, na) for b in BITS for na in (False, True)], eng.stageTimes()["radix_passes"],
                batch_shapes(eng))

    with GaussianEngine() as eng:
        eng.uploadRecords(g, 3)
        eng.setCamera(cam.view, cam.proj_view, cam.focal_ndc, cam.width, cam.height)
        view = (eng.addScene(g, Settings(3)), cam.view, cam.proj_view, cam.focal_ndc, cam.width, cam.height)
        eng.setViews([view] * 3)
        eng.setProfiling(True)
        own = shapes(eng)
        image = eng.readImage()
        for change in (lambda: eng.setSortShape(0), lambda: eng.setSortShape(9), eng.autotune, eng.autotuneBatch):
            change()
            shapes(eng)
            eng.resetSortShape()
            assert shapes(eng) == own
            assert np.array_equal(eng.readImage(), image)
            assert all(np.array_equal(eng.readBatchImage(v), image) for v in range(3))
        eng.setSortShape(0)
        assert batch_shapes(eng) == (0, 0) and not sort_in_alt(eng, 45)
