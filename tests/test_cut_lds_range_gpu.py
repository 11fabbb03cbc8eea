"""GPU test of the LDS-resident cut at the upper end of its knob: meshes around the most vertices a CU's LDS holds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _torus(n, m):
    """A torus of n x m vertices."""
    a, b = np.meshgrid(2 * np.pi * np.arange(n) / n, 2 * np.pi * np.arange(m) / m, indexing="ij")
    r = 1.0 + 0.4 * np.cos(b)
    v = np.stack([r * np.cos(a), r * np.sin(a), 0.4 * np.sin(b)], -1).reshape(-1, 3).astype(np.float32)
    i, j = np.meshgrid(np.arange(n), np.arange(m), indexing="ij")
    at = lambda x, y: (x % n) * m + y % m  # noqa: E731
    q = [at(i, j), at(i + 1, j), at(i + 1, j + 1), at(i, j + 1)]
    t = np.concatenate([np.stack([q[0], q[1], q[2]], -1).reshape(-1, 3), np.stack([q[0], q[2], q[3]], -1).reshape(-1, 3)])
    return v, t.astype(np.int32)


# 110592 vertices are the knob's most and more than fit beside the kernel's own LDS; a few thousand fewer do fit
@pytest.mark.parametrize("n,m", [(304, 330), (416, 256), (323, 330), (384, 288)])
def test_largest_knob_cuts_every_mesh_it_names(ctx, n, m):
    mesh = _torus(n, m)
    assert len(mesh[0]) <= 110592
    plane = np.array([0.6, 0.7, 0.39, 0.11], np.float32)
    old = ctx.get_tuning("cut_lds_verts")
    got = []
    try:
        for knob in (110592, 0):
            ctx.set_tuning("cut_lds_verts", knob)
            cut = ctx.plane_cut(*mesh, plane)
            batch = ctx.batch_plane_cut([mesh], [0], plane[None])
            got.append([np.asarray(x).tobytes() for x in (*cut, *batch)])
            assert min(len(x) for x in cut) > 10000
    finally:
        ctx.set_tuning("cut_lds_verts", old)
    assert got[0] == got[1]  # the same halves, bit for bit, on either path
