"""GPU tests of the cap builder at the edges of its LDS capacity: boundary loops of chosen sizes, bit for bit."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _prism(n, seed, waves):
    """A closed prism over a star-shaped n-gon (concave for waves > 0), cut across: one loop of n + n edges' points."""
    rng = np.random.default_rng(seed)
    a = np.linspace(0, 2 * np.pi, n, endpoint=False)
    r = 1.0 + (0.3 * np.sin(waves * a) if waves else 0.0) + 0.002 * rng.random(n)
    ring = np.stack([r * np.cos(a), r * np.sin(a)], 1)
    v = np.concatenate([np.c_[ring, np.zeros(n)], np.c_[ring, np.ones(n)], [[0, 0, 0], [0, 0, 1]]]).astype(np.float32)
    i, j = np.arange(n), (np.arange(n) + 1) % n
    t = np.concatenate([np.stack([i, j, j + n], 1), np.stack([i, j + n, i + n], 1),
                        np.stack([np.full(n, 2 * n), j, i], 1), np.stack([np.full(n, 2 * n + 1), i + n, j + n], 1)])
    return v, t.astype(np.int32)


def _check(ctx, v, t, plane):
    got = ctx.plane_cut(v, t, plane)
    want = oracle.plane_cut(v, t, plane)
    assert want[0] == 0
    for g, w in zip(got, want[1:]):
        assert np.asarray(g).tobytes() == np.ascontiguousarray(w, g.dtype).tobytes()


@pytest.mark.parametrize("n", [3, 31, 32, 33, 127, 128, 255, 256, 257, 300, 511, 512, 513, 700])
@pytest.mark.parametrize("waves", [0, 7])
def test_cap_of_one_loop_matches_oracle(ctx, n, waves):
    # the side walls are split by their diagonals: a horizontal cut meets 2 n edges
    v, t = _prism(n, n, waves)
    _check(ctx, v, t, np.array([0.01, -0.02, 1.0, -0.45], np.float32))


@pytest.mark.parametrize("n", [40, 300])
def test_caps_of_many_loops_match_oracle(ctx, n):
    """Several prisms in one mesh (loops side by side, and nested ones as holes)."""
    v0, t0 = _prism(n, 1, 5)
    vs, ts, o = [], [], 0
    for k, (s, dx, flip) in enumerate([(1.0, 0.0, False), (0.4, 0.0, True), (0.3, 3.0, False), (1.0, 6.0, False)]):
        v = v0 * np.float32(s)
        v[:, 2] = v0[:, 2] if not flip else 0.2 + 0.6 * v0[:, 2]
        v[:, 0] += np.float32(dx)
        vs.append(v)
        ts.append((t0[:, ::-1] if flip else t0) + o)
        o += len(v)
    _check(ctx, np.concatenate(vs), np.concatenate(ts).astype(np.int32), np.array([0.003, 0.004, 1.0, -0.47], np.float32))
