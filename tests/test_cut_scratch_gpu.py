"""GPU test of what a plane cut takes from the device pool: a pool that holds the halves and the cut's lists is enough."""
import ctypes as C
import os

import numpy as np
import pytest

from test_cut_lds_range_gpu import _torus

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _block(nbytes):
    """Pool bytes of a heap block: its 16-byte header, in size classes of powers of two."""
    return 1 << max(8, int(nbytes + 16 - 1).bit_length())


@pytest.mark.parametrize("n,m", [(2000, 24), (3500, 18), (500, 40)])
def test_cut_scratch_follows_the_special_triangles(n, m):
    lib = C.CDLL(os.path.join(ROOT, "cuacd_amd", "libcuacd_hip.so"))
    lib.gpu_init.argtypes = [C.POINTER(C.c_void_p), C.c_int, C.c_size_t]
    lib.gpu_destroy.argtypes = [C.c_void_p]
    lib.gpu_pool_usage.argtypes = [C.c_void_p]
    lib.gpu_pool_usage.restype = C.c_size_t
    lib.gpu_test_plane_cut.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_void_p, C.c_int] + [C.c_float] * 4 + \
        [C.c_void_p, C.c_int] * 4 + [C.c_void_p] * 4
    v, t = _torus(n, m)
    plane = (0.002, 1.0, 0.003, 0.0013)  # across the tube twice: a few hundred of the triangles
    cap = 2 * len(v) + 1000
    out = [np.zeros((cap * (1 + k % 2), 3), (np.float32, np.int32)[k % 2]) for k in range(4)]
    cnt = np.zeros(4, np.int32)
    ctx = C.c_void_p()
    assert lib.gpu_init(C.byref(ctx), 0, C.c_size_t(64 << 20)) == 0
    try:
        before = lib.gpu_pool_usage(ctx)
        args = [x for o in out for x in (o.ctypes.data, len(o))]
        assert lib.gpu_test_plane_cut(ctx, v.ctypes.data, len(v), t.ctypes.data, len(t), *plane, *args,
                                      *(cnt[k:].ctypes.data for k in range(4))) == 0
        used = lib.gpu_pool_usage(ctx) - before
    finally:
        lib.gpu_destroy(ctx)
    assert cnt.min() > 0
    halves = [_block((12 * int(cnt[2 * s]) + 15) // 16 * 16 + 12 * int(cnt[2 * s + 1])) for s in (0, 1)]
    # one index per triangle; the rest grows with the crossing triangles, some 4 m of them, and
    # the cap builder's with its 256 loops
    rest = _block(200 * 4 * m) + _block(200 * 4 * m + 32768)
    assert used <= sum(halves) + _block(4 * len(t) + 16) + rest, (used, halves, len(t))
