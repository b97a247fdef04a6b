"""The autotuner where a volume's launch has only a tile to choose (one workgroup
per tile), and on the two sides of such a limit within one size class."""
import numpy as np
import pytest

from lsc_helpers import synth

pytestmark = pytest.mark.gpu

LOSSLESS = ((1, 1, 1, 1), 1.0)
AXES = ("wg_per_cu", "lb_window", "counters")


@pytest.fixture
def default_shapes(gpu):
    saved = [gpu.get_launch_shape_ex(k) for k in (gpu.COMPRESS, gpu.DECOMPRESS)]
    for k in (gpu.COMPRESS, gpu.DECOMPRESS):
        gpu.set_launch_shape_ex(k, 0, 0, 0, 0)
    yield
    for k, s in zip((gpu.COMPRESS, gpu.DECOMPRESS), saved):
        gpu.set_launch_shape_ex(k, **s)


def _dev(vol):
    import torch
    return torch.from_numpy(vol.view(np.int16)).cuda()


def test_small_volume_keeps_the_axes_it_has_not(gpu, default_shapes):
    """Whatever the timings of one repetition say, a tile that runs the volume with
    one workgroup per tile comes with the workgroups per CU, window and counters
    that were set before."""
    before = [gpu.get_launch_shape_ex(k) for k in (gpu.COMPRESS, gpu.DECOMPRESS)]
    # a size class per volume; every decode here has one workgroup per tile at every tile
    for frames in (1, 2, 4, 8):
        vol = synth("sparse", (frames, 280, 280), seed=frames)
        table = gpu.autotune(_dev(vol), vol.shape, *LOSSLESS, reps=1)
        assert table
        for k, was in zip((gpu.COMPRESS, gpu.DECOMPRESS), before):
            now = gpu.get_launch_shape_ex(k)
            if k == gpu.DECOMPRESS or now["tile"] == 512:
                assert all(now[a] == was[a] for a in AXES), (k, now)
        for k in (gpu.COMPRESS, gpu.DECOMPRESS):
            gpu.set_launch_shape_ex(k, 0, 0, 0, 0)


def test_cache_keeps_kinds_of_launch_apart(gpu, default_shapes):
    """586 and 782 tiles of 512 blocks are of one size class, but only the first
    decode with one workgroup per tile: each is tuned for itself."""
    for n, cached in ((300000, False), (400000, False), (310000, True), (390000, True)):
        vol = synth("sparse", (1, 8, 8 * n), seed=5)
        table = gpu.autotune(_dev(vol), vol.shape, (7, 7, 7, 7), 0.5, reps=1)
        assert (table == []) == cached, n
