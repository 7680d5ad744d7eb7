"""Carving where blocks are new in a batch: a block is carved from the first frame of the batch whose
bands cross it, whichever frame's lane put it into the hash table first. Noisy depth, so that a block is
often crossed by a few pixels of one frame only and the frames' lanes race for it; partial tiles, both
depth formats, every storage. Bar: voxels, weights and colours identical to the oracle's, which takes
the frames one by one (no tolerance)."""
import numpy as np
import pytest

from test_gpu_color import assert_same_colour_volume
from test_gpu_integration import assert_same_volume

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,fmt,storage,color,batch", [
    (287, 211, 1, 0, 0, 8),
    (143, 97, 1, 0, 0, 3),
    (256, 160, 0, 1, 0, 8),
    (131, 113, 1, 2, 0, 0),
    (200, 96, 0, 0, 1, 8),
    (97, 65, 1, 2, 1, 5),
])
def test_blocks_new_in_a_batch(vh, oracle, W, H, fmt, storage, color, batch):
    import torch

    print(f"{W}x{H}, {'float' if fmt else 'uint16'} depth, storage {storage}, colour {color}, batch {batch}", flush=True)
    w = dict(width=W, height=H, fx=0.82 * W, fy=0.82 * W, cx=(W - 1) / 2, cy=(H - 1) / 2, min_depth=0.1, max_depth=4.0, vox_size=0.01,
             trunc=0.04, log2_buckets=17, pool_blocks=1 << 16, storage=storage, weight_cap=255 if storage else 0, color=color, carve=1)
    rng = np.random.default_rng(W)
    n = 19
    v, u = np.mgrid[0:H, 0:W]
    mm = 1400 + 500 * ((u // 31 + v // 23) % 2) + rng.normal(0, 18, (n, H, W))
    mm[rng.random((n, H, W)) < 0.02] = 0
    mm = mm.clip(0, 60000).astype(np.uint16)
    rgb = rng.integers(0, 256, (n, H, W, 3), dtype=np.uint8)
    T = np.tile(np.eye(4, dtype=np.float32), (n, 1, 1))
    for k in range(n):
        c, s = np.cos(0.006 * k), np.sin(0.006 * k)
        T[k, :3, :3] = [[c, 0, s], [0, 1, 0], [-s, 0, c]]
        T[k, :3, 3] = (0.011 * k, -0.004 * k, 0.003 * k)
    ref = oracle.Oracle(w, color=bool(color))
    for k in range(n):
        ref.integrate(mm[k], T[k], rgb=rgb[k] if color else None)
    vol = vh.Volume(vh.config_from_workload(w, seq_batch=batch))
    depth = mm.astype(np.float32) * np.float32(0.001) if fmt else mm.view(np.int16)
    d_depth, d_pose, d_rgb = torch.from_numpy(depth).cuda(), torch.from_numpy(T).cuda(), torch.from_numpy(rgb).cuda()
    torch.cuda.synchronize()
    vol.bind_sequence(d_depth, vh.DEPTH_F32 if fmt else vh.DEPTH_U16, 1.0 if fmt else 0.001, d_pose, n)
    if color:
        vol.bind_sequence_rgb(d_rgb)
    vol.integrate_next(n)
    vol.sync()
    assert vol.stats()["carved_total"] > 0
    (assert_same_colour_volume if color else assert_same_volume)(oracle, vol, ref)
    vol.close()
