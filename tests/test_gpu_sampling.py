"""The sampler, its backward pass and the solver at the edges of their lookups and launch shapes.

Cells that cross every combination of block faces, among absent and unobserved neighbours, in roomy
and in crowded hash tables (home buckets full of other keys): values and validity identical to the
oracle's. Backward over ragged point counts and several points per lane: voxel gradients identical to
a CPU scatter of inputs for which every sum is exact (lattice positions in quarters of a voxel of
2^-7 m, whole upstream values: each weight is a multiple of 1/64, each sum far below 2^24 / 64).
Solver over one and several points per lane and turn: the number of valid samples identical to the
oracle's at the starting pose, poses to the 1e-6 of the other solver tests.
"""
import numpy as np
import pytest

from conftest import look_down_z
from gn_reference import lm_reference, world_points_d

pytestmark = pytest.mark.gpu

VOX = 2.0 ** -7


def workload(storage=0, log2_buckets=14):
    return dict(width=320, height=240, fx=260.0, fy=262.0, cx=159.3, cy=119.6, min_depth=0.1, max_depth=4.0,
                vox_size=VOX, trunc=4 * VOX, log2_buckets=log2_buckets, pool_blocks=1 << 15, storage=storage,
                weight_cap=255 if storage else 0)


def scene(vh, oracle, w):
    """One view of a stepped, tilted surface with holes (so neighbours are missing or unobserved), fused twice."""
    v, u = np.mgrid[0:240, 0:320]
    d = (1100 + 2 * u + 1.5 * v + 180 * ((u // 40 + v // 30) % 2)).astype(np.uint16)
    d[(u // 16 + v // 12) % 11 == 0] = 0
    vol, ref = vh.Volume(vh.config_from_workload(w)), oracle.Oracle(w)
    for T in (look_down_z(0.0, 0.0, 0.0), look_down_z(0.01, -0.02, 0.015)):
        vol.integrate(d, T)
        ref.integrate(d, T)
    return vol, ref, d


def cells(vol, n, seed, quarters=False):
    """n world points spread over the 8 combinations of crossed block faces of the allocated blocks and their rims."""
    rng = np.random.default_rng(seed)
    keys, _, _ = vol.export_blocks()
    b = np.asarray(keys, np.int64)[rng.integers(0, len(keys), n)]
    combo = rng.integers(0, 8, n)
    cross = (combo[:, None] >> np.array([2, 1, 0])) & 1
    base = np.where(cross == 1, np.where(rng.random((n, 3)) < 0.2, -1, 7), rng.integers(0, 7, (n, 3)))
    frac = rng.integers(0, 4, (n, 3)) / 4.0 if quarters else rng.random((n, 3))
    return ((b * 8 + base + frac) * VOX).astype(np.float32)


# 2^11 buckets of four slots hold the few thousand blocks at a load where home buckets overflow
@pytest.mark.parametrize("storage,log2_buckets", [(0, 14), (1, 14), (2, 14), (0, 11), (1, 11)])
def test_cells_across_faces(vh, oracle, storage, log2_buckets):
    w = workload(storage, log2_buckets)
    vol, ref, _ = scene(vh, oracle, w)
    blocks = len(vol.export_blocks()[0])
    print(f"storage {storage}: {blocks} blocks in {4 << log2_buckets} slots", flush=True)
    for n in (1, 63, 257, 60_000):
        pts = cells(vol, n, n + storage)
        sdf, valid = vol.query(pts)
        s32, _, _, rvalid = ref.query(pts)
        assert np.array_equal(valid, rvalid)
        assert np.array_equal(sdf[valid].view(np.uint32), s32[valid].view(np.uint32))
        assert np.all(sdf[~valid] == 0)
    assert 0.05 < rvalid.mean() < 0.95
    vol.close()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 257, 5_000, 2048 * 256 - 1, 2048 * 256 + 65])
def test_backward_counts(vh, oracle, n):
    import torch

    w = workload(storage=n % 2)
    vol, ref, _ = scene(vh, oracle, w)
    pts = cells(vol, n, n, quarters=True)
    up = np.random.default_rng(n).integers(-3, 4, n).astype(np.float32)
    blocks = vol.pool_view()[2]
    grad = torch.zeros(blocks * 512, dtype=torch.float32, device="cuda")
    r = torch.empty(n, dtype=torch.float32, device="cuda")
    ok = torch.empty(n, dtype=torch.uint8, device="cuda")
    J = torch.empty(n, 6, dtype=torch.float32, device="cuda")
    pose_grad = torch.empty(6, dtype=torch.float64, device="cuda")
    d_pts, d_up = torch.from_numpy(pts).cuda(), torch.from_numpy(up).cuda()
    torch.cuda.synchronize()
    vol.backward_device(d_pts, n, np.eye(4, dtype=np.float32), d_up, r, ok, J, pose_grad, grad)
    s, g, valid = ref.query_twin(pts.astype(np.float64))
    assert np.array_equal(ok.cpu().numpy().astype(bool), valid)
    assert np.array_equal(r.cpu().numpy()[valid], s[valid])
    Jh = J.cpu().numpy()
    assert np.array_equal(Jh[:, :3][valid], g[valid]) and not Jh[~valid].any()
    terms = up.astype(np.float64)[:, None] * Jh
    # each side's FP64 sum of n products is within n 2^-53 of its terms' magnitude
    assert np.all(np.abs(pose_grad.cpu().numpy() - terms.sum(0)) <= 2 * n * 2.0 ** -53 * np.abs(terms).sum(0))
    # the scatter, block by block of the pool: voxel 8 (8 x + y) + z
    cell = np.floor(pts.astype(np.float64) / VOX).astype(np.int64)
    f = pts.astype(np.float64) / VOX - cell
    want = {}
    for k in range(8):
        o = np.array([k >> 2, (k >> 1) & 1, k & 1])
        wt = np.prod(np.where(o == 1, f, 1 - f), 1) * up
        c = cell + o
        for q, x in zip(c[valid], wt[valid]):
            want[tuple(q)] = want.get(tuple(q), 0.0) + x
    got = grad.cpu().numpy().reshape(-1, 512).astype(np.float64)
    assert got.sum() == sum(want.values()) and np.abs(got).sum() == sum(map(abs, want.values()))
    assert np.array_equal(np.sort(got[got != 0]), np.sort([x for x in want.values() if x != 0]))
    vol.close()


# partial sums: 1, 2, 129 and 512 of one point per lane; then two per lane, the second turn (over
# 3 x 131,072), a partial third
@pytest.mark.parametrize("n", [255, 257, 33_000, 131_072, 131_073, 393_217, 700_001])
def test_solver_counts(vh, oracle, n):
    w = workload()
    vol, ref, d = scene(vh, oracle, w)
    rng = np.random.default_rng(n)
    v, u = np.nonzero(d > 0)
    sel = rng.integers(0, len(v), n)
    z = d[v[sel], u[sel]] * np.float64(np.float32(0.001)) + rng.normal(0, 0.002, n)
    pts = np.stack([(u[sel] - w["cx"]) * z / w["fx"], (v[sel] - w["cy"]) * z / w["fy"], z], 1).astype(np.float32)
    pts[rng.random(n) < 0.02] = np.nan
    T0 = np.eye(4)
    T0[:3, 3] = (0.002, -0.001, 0.003)
    T, st = vol.gn_refine(pts, T0, 2)
    kept = pts[np.isfinite(pts).all(1)]
    _, _, valid = ref.query_twin(world_points_d(T0, kept))
    assert st["n_valid"][0] == valid.sum()
    want, _ = lm_reference(ref, kept, T0, 2, w["trunc"])
    assert np.abs(T - want).max() < 1e-6
    vol.close()


# 80 x 60 and 640 x 480 points of a tracked frame: one point per lane, and several; uint16 and float depth
@pytest.mark.parametrize("W,H,stride,fmt", [(320, 240, 4, 0), (320, 240, 1, 0), (640, 480, 1, 0), (640, 480, 1, 1)])
def test_tracked_frame_equals_refinement(vh, oracle, W, H, stride, fmt):
    """A tracked frame without a motion prior runs the refinement's arithmetic on its own back-projected
    points: its pose is the refinement's, rounded to FP32, bit for bit."""
    import torch

    s = W / 320
    w = dict(workload(), width=W, height=H, fx=260.0 * s, fy=262.0 * s, cx=159.3 * s, cy=119.6 * s)
    v, u = np.mgrid[0:H, 0:W]
    d = (1100 + (2 * u + 1.5 * v) / s + 180 * ((u // 40 + v // 30) % 2)).astype(np.uint16)
    d[(u // 16 + v // 12) % 11 == 0] = 0
    metres = d.astype(np.float32) * np.float32(0.001)
    a, b = (vh.Volume(vh.config_from_workload(w)) for _ in range(2))
    for vol in (a, b):
        vol.integrate(d, look_down_z(0.0, 0.0, 0.0))
    prior = look_down_z(0.002, -0.001, 0.003)
    dd = torch.from_numpy(metres if fmt else d.view(np.int16)).cuda()[None].contiguous()
    pr, out = torch.from_numpy(prior).cuda()[None].contiguous(), torch.zeros(1, 4, 4, device="cuda")
    torch.cuda.synchronize()
    a.bind_tracking(dd, vh.DEPTH_F32 if fmt else vh.DEPTH_U16, 1.0 if fmt else 0.001, 1, pr, out, None, gn_iters=4,
                    point_stride=stride)
    a.integrate_next(1)
    a.sync()
    z = metres[::stride, ::stride]
    uu, vv = (c[::stride, ::stride].astype(np.float32) for c in (u, v))
    x = ((uu - np.float32(w["cx"])) * z) / np.float32(w["fx"])
    y = ((vv - np.float32(w["cy"])) * z) / np.float32(w["fy"])
    pts = np.stack([x, y, z], -1).reshape(-1, 3)
    pts[z.reshape(-1) == 0] = np.nan
    T, _ = b.gn_refine(pts, prior, 4)
    assert np.array_equal(out.cpu().numpy()[0].view(np.uint32), T.astype(np.float32).view(np.uint32))
    a.close()
    b.close()
