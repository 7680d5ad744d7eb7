"""A host image that begins in page-locked memory and runs past its allocation into ordinary memory: the
frame's kernels read only what is mapped for the GPU whole. Bar: voxels, weights and colours identical to
the oracle's (no tolerance)."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_color import assert_same_colour_volume
from test_gpu_integration import assert_same_volume

pytestmark = pytest.mark.gpu

PAGE = 4096
libc = C.CDLL(None, use_errno=True)
libc.mmap.restype = C.c_void_p
libc.mmap.argtypes = [C.c_void_p, C.c_size_t, C.c_int, C.c_int, C.c_int, C.c_long]
libc.munmap.argtypes = [C.c_void_p, C.c_size_t]


class Straddling:
    """`bytes` at an address whose first part is the end of a page-locked allocation and whose rest is
    ordinary memory mapped right behind it."""

    def __init__(self, hip, locked, rest):
        self.hip, self.rest, self.kept, self.map = hip, -(-rest // PAGE) * PAGE, [], None
        for _ in range(16):
            p = C.c_void_p()
            assert hip.hipHostMalloc(C.byref(p), C.c_size_t(locked), C.c_uint(0)) == 0
            self.kept.append(p)
            if p.value % PAGE:
                continue
            at = libc.mmap(p.value + locked, self.rest, 3, 0x100022, -1, 0)  # private, anonymous, fixed without replacing
            if at == p.value + locked:
                self.start, self.map = p.value, at
                return
            if at and at != C.c_void_p(-1).value:
                libc.munmap(at, self.rest)

    def free(self):
        if self.map:
            libc.munmap(self.map, self.rest)
        for p in self.kept:
            assert self.hip.hipHostFree(p) == 0


def hip_runtime(vh):
    path = {line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line}
    return C.CDLL(sorted(path)[0])


@pytest.mark.parametrize("color", [0, 1])
@pytest.mark.parametrize("W,H,fmt,pad", [(128, 96, 0, 0), (127, 95, 0, 0), (96, 80, 1, 0), (96, 80, 1, 64)])
def test_image_past_its_allocation(vh, oracle, W, H, fmt, pad, color):
    print(f"{W}x{H}, {'float' if fmt else 'uint16'} depth, rows {pad} bytes apart, colour {color}", flush=True)
    w = dict(width=W, height=H, fx=0.9 * W, fy=0.9 * W, cx=W / 2 - 0.5, cy=H / 2 - 0.5, min_depth=0.1, max_depth=4.0, vox_size=0.02,
             trunc=0.08, log2_buckets=14, pool_blocks=1 << 13, storage=0, weight_cap=0, color=color)
    rng = np.random.default_rng(W)
    n = 3
    mm = (900 + rng.integers(0, 60, (n, H, W)) + 200 * np.arange(W) // W).astype(np.uint16)
    depth = mm.astype(np.float32) * np.float32(0.001) if fmt else mm
    rgb = rng.integers(0, 256, (H, W, 3), dtype=np.uint8)
    T = np.tile(np.eye(4, dtype=np.float32), (n, 1, 1))
    T[:, 0, 3] = 0.01 * np.arange(n)
    lib, ref = vh.load(), oracle.Oracle(w, color=bool(color))
    for k in range(n):
        ref.integrate(mm[k], T[k], rgb=rgb if color else None)
    row, pitch = depth[0][0].nbytes, depth[0][0].nbytes + pad
    for queued in (False, True):
        vol = vh.Volume(vh.config_from_workload(w))  # maps the runtime
        hip, mems = hip_runtime(vh), []
        span = pitch * (H - 1) + row
        for k in range(n):
            m = Straddling(hip, 1 << 16, span)
            mems.append(m)
            if not m.map:
                [x.free() for x in mems]
                vol.close()
                pytest.skip("no room behind a page-locked allocation")
            start = m.start + (1 << 16) - 8 * (span // 24)  # a third before the allocation's end, the rest behind it
            view = np.frombuffer((C.c_uint8 * span).from_address(start), np.uint8)
            for r in range(H):
                view[r * pitch : r * pitch + row] = depth[k][r].view(np.uint8)
            f = vh.Frame()
            f.depth, f.pitch = start, pitch
            f.depth_format, f.depth_scale = (vh.DEPTH_F32, 1.0) if fmt else (vh.DEPTH_U16, 0.001)
            f.c2w[:] = T[k].reshape(16).tolist()
            if color:
                f.rgb = rgb.ctypes.data
            assert (lib.vh_integrate_async if queued else lib.vh_integrate)(vol._h, C.byref(f)) == 0
        vol.sync()
        (assert_same_colour_volume if color else assert_same_volume)(oracle, vol, ref)
        vol.close()
        for m in mems:
            m.free()
