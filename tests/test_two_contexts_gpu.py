"""GPU test of two contexts on two threads: kernels are shared by the process, so what one thread sets on a kernel
(its dynamic-LDS limit) must not refuse or change the other's launches of it with other sizes."""
import ctypes as C
import os
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _lib():
    lib = C.CDLL(os.path.join(ROOT, "cuacd_amd", "libcuacd_hip.so"))
    lib.gpu_init.argtypes = [C.POINTER(C.c_void_p), C.c_int, C.c_size_t]
    lib.gpu_destroy.argtypes = [C.c_void_p]
    lib.gpu_last_error.argtypes = [C.c_void_p]
    lib.gpu_last_error.restype = C.c_char_p
    lib.gpu_hull_dandc_vol.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_void_p] + [C.c_int] * 4 + [C.c_void_p] * 6
    lib.gpu_score_cuts.argtypes = [C.c_void_p] + [C.c_void_p] * 4 + [C.c_int, C.c_void_p, C.c_void_p, C.c_int,
                                                                     C.c_float] + [C.c_void_p] * 3
    return lib


def _cloud(corners, inside, seed):
    """`corners` points of a sphere among `inside` points deep in it: what is left of it after chunking is larger
    than the sphere's share, so its last hull needs more than 8192 points."""
    rng = np.random.default_rng(seed)
    p = rng.standard_normal((corners + inside, 3))
    p /= np.linalg.norm(p, axis=1, keepdims=True)
    p[corners:] *= 0.3 * rng.random((inside, 1))
    return rng.permutation(p).astype(np.float32)


def _hull(lib, ctx, cloud):
    cap = len(cloud)
    off = np.array([0, cap], np.int32)
    v, t = np.zeros((cap, 3), np.float32), np.zeros((2 * cap, 3), np.int32)
    n = np.zeros(3, np.int32)
    vol = np.zeros(1)
    rc = lib.gpu_hull_dandc_vol(ctx, cloud.ctypes.data, cap, off.ctypes.data, 1, cap, cap, 2 * cap, v.ctypes.data,
                                t.ctypes.data, n[0:].ctypes.data, n[1:].ctypes.data, n[2:].ctypes.data,
                                vol.ctypes.data)
    return rc, n.tobytes(), v[:n[0]].tobytes(), t[:n[1]].tobytes(), vol.tobytes()


def _score(lib, ctx, mesh, planes):
    v, t = mesh
    vo, to = np.array([0, len(v)], np.int32), np.array([0, len(t)], np.int32)
    of = np.zeros(len(planes), np.int32)
    s, d = np.zeros(len(planes), np.float32), np.zeros((len(planes), 10))
    rc = lib.gpu_score_cuts(ctx, v.ctypes.data, vo.ctypes.data, t.ctypes.data, to.ctypes.data, 1,
                            of.ctypes.data, planes.ctypes.data, len(planes), 0.1,
                            s.ctypes.data, d.ctypes.data, None)
    return rc, s.tobytes(), d.tobytes()


def test_two_threads_share_kernels_with_other_sizes():
    from cuacd_amd import datasets
    lib = _lib()
    planes = np.array([[1, 0, 0, 0.05], [0, 1, 0, -0.1], [0.6, 0.8, 0, 0.02]], np.float32)
    work = []
    for k, (corners, level) in enumerate(((9000, 4), (15000, 6))):
        (mesh,) = datasets.noisy_icospheres(1, level, 0.02, seed=k)
        mesh = tuple(np.ascontiguousarray(x, d) for x, d in zip(mesh, (np.float32, np.int32)))
        work.append((_cloud(corners, 20000 - corners, k), mesh))
    ctxs = [C.c_void_p() for _ in work]
    for c in ctxs:
        assert lib.gpu_init(C.byref(c), 0, C.c_size_t(1 << 30)) == 0
    try:
        alone = [(_hull(lib, c, w[0]), _score(lib, c, w[1], planes)) for c, w in zip(ctxs, work)]
        for a in alone:
            assert a[0][0] == 0 and a[1][0] == 0, [lib.gpu_last_error(c) for c in ctxs]
        got = [[], []]

        def loop(i):
            for _ in range(6):
                got[i].append((_hull(lib, ctxs[i], work[i][0]), _score(lib, ctxs[i], work[i][1], planes)))

        threads = [threading.Thread(target=loop, args=(i,)) for i in range(2)]
        for th in threads:
            th.start()
        for th in threads:
            th.join()
        for i in range(2):
            assert len(got[i]) == 6 and all(g == alone[i] for g in got[i]), lib.gpu_last_error(ctxs[i])
    finally:
        for c in ctxs:
            lib.gpu_destroy(c)
