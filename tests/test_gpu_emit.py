"""Pair emission and the item kernel at the sizes where their partitions, alignments and records change:
frames on the GPU against the CPU oracle, sorted and unsorted pairs, ranges and images bit for bit."""
import numpy as np
import pytest

from conftest import c1_camera, small_scene
from test_gpu_forward import compare_frame

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    from torpedo_amd.engine import GaussianEngine
    e = GaussianEngine(keep_unsorted=True)
    yield e
    e.close()


# Gaussians per emission partition: 512 below 262,144 (and wherever there is room for 8 pairs each), 1,024
# below 524,288, 2,048 below 8,388,608, then 4,096; the item kernel's grid strides from 262,144 on.
@pytest.mark.parametrize("n", [1, 2, 511, 512, 513, 1023, 1024, 1025, 2049, 262_143, 262_145, 524_289])
def test_partition_edges(eng, orc, n):
    compare_frame(eng, orc, small_scene(n, seed=n, log_scale_mean=-3.5), c1_camera(orc, 200, 120), 3,
                  f"emission n={n}", check_f64=False)


@pytest.mark.parametrize("n", [1_048_577, 2_100_001, 8_388_611])
def test_larger_partitions(eng, orc, n):
    from torpedo_amd import scenes
    compare_frame(eng, orc, scenes.uniform_scene(n, seed=7, log_scale_mean=-6.0), c1_camera(orc, 640, 360), 0,
                  f"emission n={n}", check_f64=False)


@pytest.mark.parametrize("w,h", [(2032, 40), (2033, 40), (2200, 64), (32768, 16), (16, 32768)])
def test_wide_grids(eng, orc, w, h):
    """Grids of 127 (the widest whose rectangles ride in the item key) to 2048 tiles, with one Gaussian
    that covers all of them: its rectangle's width or height is the grid's."""
    from torpedo_amd.engine import gaussian_point
    g = small_scene(500, seed=w, log_scale_mean=-3.0)
    big = gaussian_point([0, 0, 0], 0.9, (0, 0, 0, 1), (4000.0,) * 3, np.full(48, 0.1, np.float32))[None]
    ref = compare_frame(eng, orc, np.concatenate([g, big]), c1_camera(orc, w, h), 3, f"grid {w}x{h}", check_f64=False)
    assert ref["splats"]["tiles"].max() == ((w + 15) // 16) * ((h + 15) // 16)


def test_rectangles_beyond_a_round(eng, orc):
    """Every Gaussian covers every tile: a block's pairs fill many rounds of 4,096 places, whose ends fall
    inside rectangles, at every alignment of the output position."""
    g = small_scene(300, seed=5, log_scale_mean=1.0)
    for w, h in [(320, 208), (333, 241)]:
        compare_frame(eng, orc, g, c1_camera(orc, w, h), 3, f"full rectangles {w}x{h}", check_f64=False)


def test_frames_of_changing_sizes(eng, orc):
    """Frames of different scenes on one engine, with tile readbacks (which scan the tile counts) between
    them: no frame may see another's look-back descriptors, counts or offsets."""
    for n, w, h in [(40_000, 320, 240), (700, 64, 48), (90_000, 500, 300), (2_500, 1000, 20), (40_000, 320, 240)]:
        compare_frame(eng, orc, small_scene(n, seed=n, log_scale_mean=-3.0), c1_camera(orc, w, h), 3,
                      f"changing n={n}", check_f64=False)
