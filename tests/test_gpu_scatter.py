"""Where the voxel gradients of the backward pass land: each voxel of the pool, found by its block's key,
holds the sum of a CPU scatter of inputs for which every sum is exact (lattice positions in quarters of a
voxel of 2^-7 m, whole upstream values: each weight is a multiple of 1/64, each sum far below 2^24 / 64).
Bar: equality, voxel by voxel; rows of the pool beyond the blocks stay as they were."""
import numpy as np
import pytest

from test_gpu_sampling import VOX, cells, scene, workload

pytestmark = pytest.mark.gpu


class Keys:
    """The pool's block keys (device memory of the volume) for torch.as_tensor."""

    def __init__(self, address, n):
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<i8", data=(address, False), version=2)


@pytest.mark.parametrize("n", [1, 63, 65, 257, 5_000, 2048 * 256 + 65])
@pytest.mark.parametrize("storage", [0, 1, 2])
def test_gradients_by_voxel(vh, oracle, n, storage):
    import torch

    print(f"{n} points, storage {storage}", flush=True)
    vol, ref, _ = scene(vh, oracle, workload(storage))
    pts = cells(vol, n, n + storage, quarters=True)
    up = np.random.default_rng(n).integers(-3, 4, n).astype(np.float32)
    _, address, blocks = vol.pool_view()
    keys = torch.as_tensor(Keys(address, blocks), device="cuda").cpu().numpy()
    grad = torch.zeros(blocks + 3, 512, dtype=torch.float32, device="cuda")
    d_pts, d_up = torch.from_numpy(pts).cuda(), torch.from_numpy(up).cuda()
    torch.cuda.synchronize()
    vol.backward_device(d_pts, n, np.eye(4, dtype=np.float32), d_up, d_voxel_grad=grad)
    _, _, valid = ref.query_twin(pts.astype(np.float64))
    cell = np.floor(pts.astype(np.float64) / VOX).astype(np.int64)
    f = pts.astype(np.float64) / VOX - cell
    order = np.argsort(keys)
    want = np.zeros((blocks + 3, 512))
    for k in range(8):
        o = np.array([k >> 2, (k >> 1) & 1, k & 1])
        weight = np.prod(np.where(o == 1, f, 1 - f), 1) * up
        at = cell + o
        b = (at >> 3) + (1 << 20)
        key = b[:, 0] << 42 | b[:, 1] << 21 | b[:, 2]
        place = order[np.searchsorted(keys, key, sorter=order).clip(max=blocks - 1)]
        assert np.array_equal(keys[place[valid]], key[valid])
        voxel = ((at[:, 0] & 7) * 8 + (at[:, 1] & 7)) * 8 + (at[:, 2] & 7)
        np.add.at(want, (place[valid], voxel[valid]), weight[valid])
    assert np.array_equal(grad.cpu().numpy().astype(np.float64), want)
    vol.close()
