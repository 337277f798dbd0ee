"""Frames and batches of changing scenes, sizes, depths and pair counts with the launch shapes the library
chooses itself: the tests of other modules whose engines are left with a selected shape by then, run here on
engines that never had one."""
import pytest

from test_gpu_batch import (test_back_to_back_steps_after_an_overflow, test_batch_all_items_culled,  # noqa: F401
                            test_batch_backward_equals_sum_of_plain, test_batch_camera_update_and_growth,
                            test_batch_emission_of_large_footprints, test_batch_entities_with_transforms,
                            test_batch_uneven_scenes, test_batch_without_gaussians, test_two_frames_in_flight)
from test_gpu_forward import (test_bind_device_scene_after_an_entity_upload, test_buffer_growth_replay,  # noqa: F401
                              test_cluster_scene_1m_1080p, test_entities_and_transforms)

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    from torpedo_amd.engine import GaussianEngine
    e = GaussianEngine(keep_unsorted=True)
    yield e
    e.close()


@pytest.fixture(scope="module")
def engines():
    from torpedo_amd.engine import GaussianEngine
    b, p = GaussianEngine(), GaussianEngine()
    yield b, p
    b.close()
    p.close()
