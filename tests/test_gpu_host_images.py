"""Host frames by every way their images reach the device: pageable and page-locked memory, rows
together and pitched (whole words apart and not), even and odd widths, both depth formats, with
colours, synchronous and queued (more frames than ring slots). Bar: voxels, weights and colours identical to
the oracle's (no tolerance)."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_color import assert_same_colour_volume
from test_gpu_integration import assert_same_volume

pytestmark = pytest.mark.gpu


def workload(W, H, color):
    return dict(width=W, height=H, fx=0.9 * W, fy=0.9 * W, cx=W / 2 - 0.5, cy=H / 2 - 0.5, min_depth=0.1, max_depth=4.0,
                vox_size=0.02, trunc=0.08, log2_buckets=14, pool_blocks=1 << 13, storage=0, weight_cap=0, color=color)


def image(a, pitch, locked, shift):
    """The rows of a, `pitch` bytes apart and `shift` bytes into their buffer: (address, what keeps it)."""
    import torch

    H, row = a.shape[0], a[0].nbytes
    buf = torch.zeros(H * pitch + 16, dtype=torch.uint8, pin_memory=locked)
    view = buf.numpy()[shift : shift + H * pitch].reshape(H, pitch)
    view[:, :row] = a.reshape(H, -1).view(np.uint8)
    view[:, row:] = 0xAB  # never read
    return buf.data_ptr() + shift, buf


@pytest.mark.parametrize("locked", [False, True])
@pytest.mark.parametrize("W,H,fmt,pad,shift", [(64, 48, 0, 0, 0), (63, 47, 0, 0, 0), (63, 47, 0, 2, 0), (62, 33, 0, 6, 2),
                                               (64, 48, 0, 64, 0), (61, 40, 1, 0, 0), (61, 40, 1, 12, 0)])
def test_host_images(vh, oracle, W, H, fmt, pad, shift, locked):
    color = (W + pad) % 2
    w = workload(W, H, color)
    rng = np.random.default_rng(W * 100 + pad)
    n = 7
    mm = (900 + rng.integers(0, 60, (n, H, W)) + 4 * np.arange(W)).astype(np.uint16)
    mm[rng.random((n, H, W)) < 0.05] = 0
    depth = mm.astype(np.float32) * np.float32(0.001) if fmt else mm
    rgb = rng.integers(0, 256, (n, H, W, 3), dtype=np.uint8)
    T = np.tile(np.eye(4, dtype=np.float32), (n, 1, 1))
    T[:, 0, 3] = 0.01 * np.arange(n)
    lib, ref = vh.load(), oracle.Oracle(w, color=bool(color))
    for k in range(n):
        ref.integrate(mm[k], T[k], rgb=rgb[k] if color else None)
    for queued in (False, True):
        vol, keep = vh.Volume(vh.config_from_workload(w)), []
        for k in range(n):
            f = vh.Frame()
            f.depth, b = image(depth[k], depth[k][0].nbytes + pad, locked, shift)
            f.pitch = 0 if pad == 0 and k % 2 else depth[k][0].nbytes + pad
            f.depth_format, f.depth_scale = (vh.DEPTH_F32, 1.0) if fmt else (vh.DEPTH_U16, 0.001)
            f.c2w[:] = T[k].reshape(16).tolist()
            if color:
                f.rgb, c = image(rgb[k], 3 * W, locked, shift)
                keep.append(c)
            keep.append(b)
            assert (lib.vh_integrate_async if queued else lib.vh_integrate)(vol._h, C.byref(f)) == 0
        vol.sync()
        assert vol.stats()["frames"] == n
        (assert_same_colour_volume if color else assert_same_volume)(oracle, vol, ref)
        vol.close()


@pytest.mark.parametrize("locked", [False, True])
def test_images_on_both_sides_of_the_direct_copy(vh, oracle, locked):
    """700 x 600: uint16 is read in the frame's own stream, float32 (1.68 MB) copied on the other one; the
    queue takes runs of both, so that slots change hands both ways."""
    import torch

    W, H = 700, 600
    w = workload(W, H, 0)
    rng = np.random.default_rng(3)
    kinds = [0, 1, 1, 0, 0, 1, 1, 1, 1, 1, 1, 0, 0, 0, 0, 0, 1]
    base = (1000 + 0.5 * np.arange(W) + 0.3 * np.arange(H)[:, None]).astype(np.uint16)
    mm = [(base + rng.integers(0, 30, (H, W)).astype(np.uint16)) for _ in kinds]
    vol, ref, keep = vh.Volume(vh.config_from_workload(w)), oracle.Oracle(w), []
    T = np.eye(4, dtype=np.float32)
    for k, d in zip(kinds, mm):
        ref.integrate(d, T)
        a = torch.from_numpy(d.astype(np.float32) * np.float32(0.001) if k else d.view(np.int16))
        keep.append(a.pin_memory() if locked else a)
        vol.integrate_async(keep[-1], T)
    vol.sync()
    assert vol.stats()["frames"] == len(kinds)
    assert_same_volume(oracle, vol, ref)
    vol.close()
