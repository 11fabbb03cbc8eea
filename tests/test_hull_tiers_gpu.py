"""GPU tests of the batch hull entry's size tiers: one call over every tier's edges, retries and packed readback."""
import numpy as np
import pytest

import lookahead_oracle as LO

pytestmark = pytest.mark.gpu

SIZES = (3, 4, 512, 513, 700, 1024, 1025, 2048, 2049, 4096, 4097, 8192, 8193, 9001)


def _sphere(n, seed):
    p = np.random.default_rng(seed).standard_normal((n, 3))
    return (p / np.linalg.norm(p, axis=1, keepdims=True)).astype(np.float32)


@pytest.mark.parametrize("kind", ["ball", "sphere", "lattice"])
def test_every_tier_in_one_call_matches_oracle(ctx, kind):
    clouds = []
    for n in SIZES:
        if kind == "lattice":
            clouds.append(np.random.default_rng(n).integers(0, 9, (n, 3)).astype(np.float32))
        else:
            r = np.random.default_rng(n).random((n, 1)) ** (1.0 / 3.0) if kind == "ball" else 1.0
            clouds.append((_sphere(n, n) * r).astype(np.float32))
    # on a sphere nearly every point is a corner: the LDS tiers overflow into their retries
    for n, c, (hv, ht, vol) in zip(SIZES, clouds, ctx.batch_hull_dandc_mesh(clouds)):
        ev, et, evol = LO.hull_mesh(c)
        assert hv.tobytes() == np.asarray(ev, np.float32).tobytes(), n
        assert np.array_equal(ht, et), n
        assert abs(vol - evol) <= 1e-12 * max(abs(evol), 1e-30), n


def test_cloud_above_the_stated_maximum_reports_capacity(ctx):
    """A device caller whose max_pts understates a cloud gets an error for it and right hulls beside it."""
    from cuacd_amd import _gpu
    clouds = [_sphere(n, n) for n in (100, 300, 900)]
    off = np.zeros(4, np.int32)
    off[1:] = np.cumsum([len(c) for c in clouds])
    pts = np.concatenate(clouds)
    m, mt = 900, 1796
    host = [np.zeros(s, d) for s, d in ((3, np.int32), (3, np.int32), (3, np.int32))]
    sizes = [pts.nbytes, off.nbytes, 3 * m * 12, 3 * mt * 12, 12, 12, 12, 24]
    bufs = [_gpu.dev_alloc(b) for b in sizes]
    try:
        _gpu.memcpy_h2d(bufs[0], pts.ctypes.data, pts.nbytes)
        _gpu.memcpy_h2d(bufs[1], off.ctypes.data, off.nbytes)
        _gpu.hull_dandc_dev(bufs[0], bufs[1], 3, 128, m, mt, *bufs[2:])
        _gpu.sync()
        for h, b in zip(host, bufs[4:7]):
            _gpu.memcpy_d2h(h.ctypes.data, b, h.nbytes)
    finally:
        for b in bufs:
            _gpu.dev_free(b)
    nv, nt, err = host
    assert nv[0] == len(LO.hull_mesh(clouds[0])[0]) and err[0] == 0
    assert err[1] != 0 and err[2] != 0


@pytest.mark.parametrize("kind", ["disc", "twice"])
@pytest.mark.parametrize("n", [600, 1500, 4000, 9000])
def test_multi_apex_rounds_at_their_limits_match_oracle(ctx, kind, n):
    """A region of more faces than the LDS lists hold; points of one grid position owned by different waves."""
    if kind == "disc":
        a = np.random.default_rng(n).permutation(n - 2) * (2 * np.pi / (n - 2))
        c = np.stack([np.cos(a), np.sin(a), np.zeros_like(a)], 1)
        c = np.concatenate([c, [[0.0, 0.0, 3 / 5108], [0.1, 0.0, -1 / 5108]]]).astype(np.float32)
    else:
        half = _sphere(n // 2, n).astype(np.float64)
        order = np.random.default_rng(n).permutation(2 * len(half))
        c = np.concatenate([half, half * (1 - 1e-6)])[order].astype(np.float32)
    (hv, ht, vol), = ctx.batch_hull_dandc_mesh([c])
    ev, et, evol = LO.hull_mesh(c)
    assert hv.tobytes() == np.asarray(ev, np.float32).tobytes()
    assert np.array_equal(ht, et)
    assert abs(vol - evol) <= 1e-12 * max(abs(evol), 1e-30)
