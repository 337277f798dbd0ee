"""The blend's tile order where its way of counting changes: one block's 1,024 tiles, the four blocks that
each count all tiles, and the first frame beyond."""
import pytest

import test_gpu_forward

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    from torpedo_amd.engine import GaussianEngine
    e = GaussianEngine()
    yield e
    e.close()


@pytest.mark.parametrize("w,h", [(16, 16), (512, 512), (512, 513), (1024, 1024), (1040, 1024)])
def test_order_of(eng, orc, w, h):
    test_gpu_forward.test_tile_order_is_a_heaviest_first_permutation(eng, orc, w, h)
