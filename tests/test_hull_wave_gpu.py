"""GPU tests of the one-wave quickhull: canonical meshes equal to the oracle's at the edges of its sizes."""
import numpy as np
import pytest

import lookahead_oracle as LO

pytestmark = pytest.mark.gpu

KINDS = ("ball", "sphere", "lattice", "cap", "cone")


def _cloud(kind, n, seed):
    rng = np.random.default_rng(seed)
    if kind == "lattice":  # coplanar, collinear and repeated points
        return rng.integers(0, 2 + int(round(n ** 0.4)), (n, 3)).astype(np.float32)
    p = rng.standard_normal((n, 3))
    p /= np.linalg.norm(p, axis=1, keepdims=True)
    if kind == "ball":
        p *= rng.random((n, 1)) ** (1.0 / 3.0)
    if kind in ("cap", "cone"):
        # a cap of the sphere seen from one far point (last or first): that
        # point's insertion replaces a region of more than 64 faces by a cone
        # over more than 64 horizon edges
        p[:, 2] = 1.0 - 0.05 * np.abs(p[:, 2])
        p[:, :2] *= np.sqrt(np.maximum(1.0 - p[:, 2:] ** 2, 0)) / np.linalg.norm(p[:, :2], axis=1, keepdims=True)
        if kind == "cone":  # a ring: every point is on the horizon of the apex
            t = np.linspace(0, 2 * np.pi, n, endpoint=False)
            p = np.stack([np.cos(t), np.sin(t), 0.05 * rng.random(n)], 1)
        p[-1] = (0.01, 0.02, 3.0)
        p[0] = (0.0, 0.01, -3.0)
    return p.astype(np.float32)


@pytest.mark.parametrize("n", [4, 5, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1024])
def test_wave_hull_matches_oracle_at_tier_edges(ctx, n):
    clouds = [_cloud(k, n, 7 * n + i) for i, k in enumerate(KINDS)]
    for kind, c, (hv, ht, vol) in zip(KINDS, clouds, ctx.batch_hull_dandc_mesh(clouds)):
        ev, et, evol = LO.hull_mesh(c)
        assert hv.tobytes() == np.asarray(ev, np.float32).tobytes(), kind
        assert np.array_equal(ht, et), kind
        if len(et):
            assert abs(vol - evol) <= 1e-12 * max(abs(evol), 1e-30), kind
