"""Queued host frames at the size where their way to the device changes: 640 x 512 uint16 (640 KB) is the largest
read in the frame's own stream from page-locked memory, one column more and float32 go by the copy stream, rows of
whole words and not; from pageable memory both are read there (up to 1.6 MB). Runs of both formats and, mixed, of both
memories, so that slots change hands every way. Bar: voxels and weights identical to the oracle's."""
import numpy as np
import pytest

from test_gpu_host_images import workload
from test_gpu_integration import assert_same_volume

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("locked", ["none", "all", "mixed"])
@pytest.mark.parametrize("W", [640, 641])
def test_both_ways_in_one_queue(vh, oracle, W, locked):
    import torch

    H = 512
    w = workload(W, H, 0)
    rng = np.random.default_rng(W)
    kinds = [0, 0, 1, 1, 0, 1, 0, 0, 0, 0, 0, 1, 1, 1, 1, 1, 0]
    base = (1000 + 0.5 * np.arange(W) + 0.3 * np.arange(H)[:, None]).astype(np.uint16)
    vol, ref, keep = vh.Volume(vh.config_from_workload(w)), oracle.Oracle(w), []
    T = np.eye(4, dtype=np.float32)
    for j, k in enumerate(kinds):
        d = base + rng.integers(0, 30, (H, W)).astype(np.uint16)
        ref.integrate(d, T)
        a = torch.from_numpy(d.astype(np.float32) * np.float32(0.001) if k else d.view(np.int16))
        keep.append(a.pin_memory() if locked == "all" or (locked == "mixed" and j % 3) else a)
        vol.integrate_async(keep[-1], T)
    vol.sync()
    assert vol.stats()["frames"] == len(kinds)
    assert_same_volume(oracle, vol, ref)
    vol.close()
