"""Batched integration against the oracle at the edges of its fast form: image widths around the
16-byte row pitch, windows from a few pixels to more than a wave's LDS window, blocks at the image
border, weight caps around the end of the reciprocal table (1,023), launches of 8 and of 1, 2 and 3
frames, and sequences that pass the table's end. Bar: voxels bit-identical (no tolerance)."""
import numpy as np
import pytest

from test_gpu_integration import assert_same_volume

pytestmark = pytest.mark.gpu


def workload(W, H, fx, storage, cap):
    return dict(width=W, height=H, fx=fx, fy=fx, cx=(W - 1) / 2 + 0.25, cy=(H - 1) / 2 - 0.5, min_depth=0.1, max_depth=3.0,
                vox_size=0.01, trunc=0.04, log2_buckets=14, pool_blocks=1 << 14, storage=storage, weight_cap=cap)


def frames(W, H, n, seed):
    """A stepped surface between 0.2 and 1.6 m with noise and holes, under small camera motions."""
    rng = np.random.default_rng(seed)
    v, u = np.mgrid[0:H, 0:W]
    base = 200 + 1400 * ((u // max(1, W // 5) + v // max(1, H // 3)) % 4) / 3
    d = base[None] + rng.normal(0, 4, (n, H, W))
    d[rng.random((n, H, W)) < 0.03] = 0
    T = np.zeros((n, 4, 4), np.float32)
    for k in range(n):
        a = 0.02 * k + 0.1
        T[k] = np.eye(4)
        T[k, :3, :3] = [[np.cos(a), 0, np.sin(a)], [0, 1, 0], [-np.sin(a), 0, np.cos(a)]]
        T[k, :3, 3] = (0.01 * (k % 7), -0.005 * (k % 5), 0.3)
    return d.clip(0, 4000).astype(np.uint16), T


def run(vh, oracle, w, depth, T, **over):
    import torch

    vol = vh.Volume(vh.config_from_workload(w, **over))
    ref = oracle.Oracle(w, storage=w["storage"], weight_cap=w["weight_cap"], shadow=True)
    touched = sum(ref.integrate(depth[k], T[k]) for k in range(len(depth)))
    dd = torch.from_numpy(depth.view(np.int16)).cuda()
    pp = torch.from_numpy(T).cuda()
    torch.cuda.synchronize()
    vol.bind_sequence(dd, vh.DEPTH_U16, 0.001, pp, len(depth))
    vol.integrate_next(len(depth))
    vol.sync()
    assert vol.stats()["touched_total"] == touched
    assert_same_volume(oracle, vol, ref)
    vol.close()


@pytest.mark.parametrize("size", [(61, 47, 60.0), (64, 48, 250.0), (129, 37, 110.0), (34, 90, 30.0)])
@pytest.mark.parametrize("storage,cap", [(0, 0), (0, 5), (1, 7), (2, 9)])
def test_batches_at_odd_sizes(vh, oracle, size, storage, cap):
    W, H, fx = size
    depth, T = frames(W, H, 19, W + storage)
    print(f"{W}x{H} fx {fx} storage {storage} cap {cap}: batches of 8, 8, 3", flush=True)
    run(vh, oracle, workload(W, H, fx, storage, cap), depth, T)


@pytest.mark.parametrize("batch", [1, 2, 3])
def test_small_batches(vh, oracle, batch):
    depth, T = frames(61, 47, 7, batch)
    print(f"61x47, batches of {batch}", flush=True)
    run(vh, oracle, workload(61, 47, 60.0, 0, 0), depth, T, seq_batch=batch)


@pytest.mark.parametrize("storage,cap", [(0, 0), (0, 1021), (0, 1022), (0, 1023), (1, 1022), (1, 1030)])
def test_weights_around_the_table_end(vh, oracle, storage, cap):
    depth, T = frames(24, 20, 13, 5)
    depth, T = np.concatenate([depth] * 81), np.concatenate([T] * 81)  # 1,053 frames
    print(f"24x20, {len(depth)} frames, storage {storage}, cap {cap}", flush=True)
    run(vh, oracle, workload(24, 20, 25.0, storage, cap), depth, T)
