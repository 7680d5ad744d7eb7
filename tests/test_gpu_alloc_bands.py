"""Allocation against the oracle over the forms its tile pass takes: bands of a fraction of a block to
several blocks (one key, closed form, walk in the window, walk block by block), keys of small and
large block coordinates (small voxels, scaled poses), poses at and far from the origin and
on block faces, single frames and batches, images of partial tiles. Bar: per-frame touched counts,
allocated sets and voxels identical (no tolerance)."""
import numpy as np
import pytest

from test_gpu_integration import assert_same_volume

pytestmark = pytest.mark.gpu


def workload(W, H, vox, trunc, max_depth=4.0):
    f = 0.8 * W
    return dict(width=W, height=H, fx=f, fy=f * 1.02, cx=(W - 1) / 2, cy=(H - 1) / 2 + 0.4, min_depth=0.1, max_depth=max_depth,
                vox_size=vox, trunc=trunc, log2_buckets=17, pool_blocks=1 << 17, storage=0, weight_cap=0)


def frames(W, H, n, seed, shift, scale=1.0):
    rng = np.random.default_rng(seed)
    v, u = np.mgrid[0:H, 0:W]
    d = 900 + 5 * u + 8 * v + 1200 * ((u + v) // 23 % 3 == 0) + rng.normal(0, 12, (n, H, W))
    d[rng.random((n, H, W)) < 0.05] = 0
    T = np.zeros((n, 4, 4), np.float32)
    for k in range(n):
        if k == 0:  # axis-aligned, so that many coordinates and crossings coincide
            R = np.eye(3)
        else:
            R = np.linalg.qr(rng.normal(0, 1, (3, 3)))[0]
            R *= np.sign(np.linalg.det(R))
        T[k] = np.eye(4)
        T[k, :3, :3] = R * scale
        T[k, :3, 3] = np.asarray(shift) + rng.normal(0, 0.05, 3) * (k > 0)
    return d.clip(0, 60000).astype(np.uint16), T


def check(vh, oracle, w, depth, T):
    import torch

    n = len(depth)
    ref = oracle.Oracle(w)
    single = vh.Volume(vh.config_from_workload(w))
    total = 0
    for k in range(n):
        touched = ref.integrate(depth[k], T[k])
        single.integrate(depth[k], T[k])
        assert single.stats()["touched_last"] == touched, k
        total += touched
    assert_same_volume(oracle, single, ref)
    single.close()
    batch = vh.Volume(vh.config_from_workload(w))
    dd, pp = torch.from_numpy(depth.view(np.int16)).cuda(), torch.from_numpy(T).cuda()
    torch.cuda.synchronize()
    batch.bind_sequence(dd, vh.DEPTH_U16, 0.001, pp, n)
    batch.integrate_next(n)
    batch.sync()
    assert batch.stats()["touched_total"] == total
    assert_same_volume(oracle, batch, ref)
    batch.close()


@pytest.mark.parametrize("trunc_voxels", [0.5, 2, 4, 5, 8, 12, 30])
@pytest.mark.parametrize("size", [(80, 60), (67, 33)])
def test_band_lengths(vh, oracle, trunc_voxels, size):
    W, H = size
    print(f"{W}x{H}, band of +-{trunc_voxels} voxels", flush=True)
    depth, T = frames(W, H, 5, int(10 * trunc_voxels), (0.3, -0.2, 0.1))
    check(vh, oracle, workload(W, H, 0.02, 0.02 * trunc_voxels), depth, T)


@pytest.mark.parametrize("vox,shift,scale", [
    (0.02, (0.0, 0.0, 0.0), 1.0),          # the camera on a block corner
    (0.02, (0.16 * 7, -0.16 * 3, 0.0), 1.0),  # and on others
    (0.02, (2000.0, -1500.0, 900.0), 1.0),  # coarse coordinates
    (0.0011, (0.2, 0.1, -0.3), 1.0),       # block coordinates in the hundreds
    (0.02, (0.3, 0.2, 0.1), 3.0),          # rows longer than a rotation's
])
def test_keys_and_poses(vh, oracle, vox, shift, scale):
    print(f"voxel {vox}, camera at {shift}, pose scale {scale}", flush=True)
    depth, T = frames(48, 40, 4, 3, shift, scale)
    check(vh, oracle, workload(48, 40, vox, 4 * vox), depth, T)
