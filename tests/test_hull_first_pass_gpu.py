"""GPU tests of the one-wave hull tiers' reduced-capacity first pass and its retries, in the host-counted hull call."""
import numpy as np
import pytest

import lookahead_oracle as LO

pytestmark = pytest.mark.gpu


def _clouds(lo, hi, n):
    """Sets of lo..hi points, a third of them on a sphere (every point a corner: past any reduced capacity), a third
    balls (few corners) and a third lattices (coplanar, collinear and repeated points)."""
    out = []
    for i in range(n):
        rng = np.random.default_rng(1000 * hi + i)
        m = (lo, hi)[i] if i < 2 else int(rng.integers(lo, hi + 1))
        p = rng.standard_normal((m, 3))
        p /= np.linalg.norm(p, axis=1, keepdims=True)
        if i % 3 == 1:
            p *= rng.random((m, 1)) ** (1.0 / 3.0)
        elif i % 3 == 2:
            p = rng.integers(0, 9, (m, 3))
        out.append(p.astype(np.float32))
    return out


def _same(got, want):
    return all(a[0].tobytes() == b[0].tobytes() and np.array_equal(a[1], b[1]) and a[2] == b[2]
               for a, b in zip(got, want))


# a tier takes a first pass when it holds more sets than the device has room for at full capacity: five to a CU of
# 129-256 points, two of 257-512 (256 CUs); hull_wide_min 256 sends the larger tier to the four- and eight-wave kernels
@pytest.mark.parametrize("lo,hi,n", [(129, 256, 1600), (257, 512, 800)])
def test_first_pass_and_retries_match_oracle(ctx, lo, hi, n):
    clouds = _clouds(lo, hi, n)
    got = ctx.batch_kdop_hull_mesh(clouds)
    for i, (c, (hv, ht, vol)) in enumerate(zip(clouds, got)):
        ev, et, evol = LO.hull_mesh(c)
        assert hv.tobytes() == np.asarray(ev, np.float32).tobytes(), i
        assert np.array_equal(ht, et), i
        assert abs(vol - evol) <= 1e-6 * max(abs(evol), 1e-30), i  # FP32 on the way out
    start = ctx.get_tuning()
    try:
        for var in ({"hull_half_cap": 0}, {"hull_vcap_eighths": 1}, {"hull_vcap_eighths": 7}, {"hull_wide_min": 0},
                    {"hull_wide_min": 256, "hull_w8": 0}, {"hull_wide_min": 256, "hull_w8": 10},
                    {"hull_wide_min": 128, "hull_w8": 15}):
            for k, v in {**start, **var}.items():
                ctx.set_tuning(k, v)
            assert _same(ctx.batch_kdop_hull_mesh(clouds), got), var
    finally:
        for k, v in start.items():
            ctx.set_tuning(k, v)


def test_fewer_sets_than_the_device_holds_take_one_pass(ctx):
    """The same sets in a small call (no first pass) and in a large one give the same bits."""
    clouds = _clouds(257, 512, 800)
    assert _same(ctx.batch_kdop_hull_mesh(clouds)[:60], ctx.batch_kdop_hull_mesh(clouds[:60]))


@pytest.mark.parametrize("wide_min", [0, 512])
def test_score_plan_keeps_its_hull_kernels(ctx, wide_min):
    """A plan's device-counted hull call has no one-wave first passes, and the knob cannot ask for them: its replays
    give the eager scores (several replays, with eager work between them)."""
    from cuacd_amd import datasets, sdf
    meshes = sdf.sdf_meshes(3, seed=9, res=48, min_tris=2000, max_tris=40000)
    planes = [datasets.cut_candidates(v, t, n_edges=6, n_total=16, seed=m) for m, (v, t) in enumerate(meshes)]
    mesh_of = np.concatenate([np.full(len(p), m, np.int32) for m, p in enumerate(planes)])
    planes = np.concatenate(planes)
    start = ctx.get_tuning()
    try:
        ctx.set_tuning("hull_wide_min", wide_min)
        eager, detail, _ = ctx.batch_score_cuts(meshes, mesh_of, planes, threshold=0.1, return_detail=True)
        plan = ctx.score_plan(meshes, mesh_of, planes, threshold=0.1)
        for _ in range(3):
            s, d = plan.run(return_detail=True)
            assert np.array_equal(s, eager) and np.array_equal(d, detail)
            assert np.array_equal(ctx.batch_score_cuts(meshes, mesh_of, planes, threshold=0.1)[:4], eager[:4])
        plan.close()
    finally:
        for k, v in start.items():
            ctx.set_tuning(k, v)
