"""Frames of a bound sequence one at a time, each a launch of its own whose blocks are placed one by one: odd
sizes, windows from a few pixels to more than a wave's LDS window, blocks at the image border, every
storage, colour. Bar: voxels and colours bit-identical to the oracle's (no tolerance)."""
import numpy as np
import pytest

from test_gpu_batch_update import frames, workload
from test_gpu_color import assert_same_colour_volume
from test_gpu_integration import assert_same_volume

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(61, 47, 60.0), (64, 48, 250.0), (129, 37, 110.0), (34, 90, 30.0), (3, 5, 8.0)])
@pytest.mark.parametrize("storage,cap,color", [(0, 0, 0), (0, 5, 1), (1, 7, 0), (2, 9, 0), (2, 9, 1)])
def test_one_frame_a_launch(vh, oracle, size, storage, cap, color):
    import torch

    W, H, fx = size
    n = 9
    depth, T = frames(W, H, n, W + storage)
    rgb = np.random.default_rng(W).integers(0, 256, (n, H, W, 3), dtype=np.uint8)
    print(f"{W}x{H} fx {fx} storage {storage} cap {cap} colour {color}: one frame a launch", flush=True)
    w = dict(workload(W, H, fx, storage, cap), color=color)
    vol, ref = vh.Volume(vh.config_from_workload(w)), oracle.Oracle(w, color=bool(color))
    d_depth, d_pose, d_rgb = torch.from_numpy(depth.view(np.int16)).cuda(), torch.from_numpy(T).cuda(), torch.from_numpy(rgb).cuda()
    torch.cuda.synchronize()
    vol.bind_sequence(d_depth, vh.DEPTH_U16, 0.001, d_pose, n)
    if color:
        vol.bind_sequence_rgb(d_rgb)
    for k in range(n):
        ref.integrate(depth[k], T[k], rgb=rgb[k] if color else None)
        vol.integrate_next(1)
    vol.sync()
    (assert_same_colour_volume if color else assert_same_volume)(oracle, vol, ref)
    vol.close()
