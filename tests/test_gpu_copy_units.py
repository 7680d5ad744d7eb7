"""Host images read by the kernel in units of 8 bytes with the bytes before and after apart: every
alignment of page-locked images, from a single pixel up, one frame at a time and queued into slots
that start at any byte. Bar: voxels, weights and colours identical to the oracle's (no tolerance)."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_color import assert_same_colour_volume

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(1, 1), (3, 1), (1, 5), (5, 3), (33, 31), (129, 65)])
def test_alignments(vh, oracle, W, H):
    import torch

    print(f"{W}x{H}", flush=True)
    w = dict(width=W, height=H, fx=0.9 * W + 3, fy=0.9 * W + 3, cx=W / 2 - 0.5, cy=H / 2 - 0.5, min_depth=0.1, max_depth=4.0,
             vox_size=0.02, trunc=0.08, log2_buckets=13, pool_blocks=1 << 12, storage=0, weight_cap=0, color=1)
    rng = np.random.default_rng(W)
    n = 9
    mm = (900 + rng.integers(0, 60, (n, H, W))).astype(np.uint16)
    rgb = rng.integers(0, 256, (n, H, W, 3), dtype=np.uint8)
    T = np.tile(np.eye(4, dtype=np.float32), (n, 1, 1))
    T[:, 0, 3] = 0.01 * np.arange(n)
    lib, ref = vh.load(), oracle.Oracle(w, color=True)
    for k in range(n):
        ref.integrate(mm[k], T[k], rgb=rgb[k])
    for queued in (False, True):
        vol, keep = vh.Volume(vh.config_from_workload(w)), []

        def locked(a, shift):
            buf = torch.zeros(a.nbytes + 16, dtype=torch.uint8, pin_memory=True)
            buf.numpy()[shift : shift + a.nbytes] = a.reshape(-1).view(np.uint8)
            keep.append(buf)
            return buf.data_ptr() + shift

        for k in range(n):
            f = vh.Frame()
            f.depth, f.rgb = locked(mm[k], k % 8 & ~1), locked(rgb[k], (3 * k) % 8)
            f.depth_format, f.depth_scale = vh.DEPTH_U16, 0.001
            f.c2w[:] = T[k].reshape(16).tolist()
            assert (lib.vh_integrate_async if queued else lib.vh_integrate)(vol._h, C.byref(f)) == 0
        vol.sync()
        assert_same_colour_volume(oracle, vol, ref)
        vol.close()
