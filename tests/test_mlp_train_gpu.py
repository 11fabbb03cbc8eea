"""GPU tests of the fused training step: gradients against the FP64 oracle at the edges of its row groups."""
import numpy as np
import pytest

from cuacd_amd import proposal as PR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,P,side", [(1, 1, "mixed"), (2, 1, "pos"), (15, 2, "neg"), (16, 1, "mixed"),
                                      (17, 3, "mixed"), (64, 4, "neg"), (65, 5, "mixed"), (300, 7, "mixed")])
@pytest.mark.parametrize("repeat", [False, True])
def test_gradients_match_oracle_at_group_edges(ctx, C, P, side, repeat):
    """Candidate counts around 16, planes with one side empty, and samples that repeat (ties in the max-pool:
    the first sample takes the gradient, as in the oracle)."""
    import mlp_oracle as MO
    rng = np.random.default_rng(C + 100 * P)
    pts = rng.uniform(-1, 1, (P, MO.NS, 3)).astype(np.float32)
    if repeat:
        pts[:, 128:] = pts[:, :128]
    planes = rng.normal(size=(C, 4)).astype(np.float32)
    planes[:, :3] /= np.linalg.norm(planes[:, :3], axis=1, keepdims=True)
    if side != "mixed":
        planes[:, 3] = 3.0 if side == "pos" else -3.0
    part_of = np.sort(rng.integers(0, P, C)).astype(np.int32)
    t = rng.uniform(0, 1, C).astype(np.float32)
    net = PR.ProposalNet(ctx, seed=3)
    try:
        params = net.params().astype(np.float64)
        loss_ref, g_ref, _ = MO.loss_and_grads(params, pts, planes, part_of, t)
        loss, g = net.train_step(pts, planes, part_of, t, apply=False, return_grads=True)
        again = net.train_step(pts, planes, part_of, t, apply=False, return_grads=True)[1]
    finally:
        net.close()
    assert np.array_equal(g, again)  # fixed summation order
    assert abs(loss - loss_ref) <= 1e-3 * loss_ref + 1e-6
    gd, rd = MO.unpack(g.astype(np.float64)), MO.unpack(g_ref)
    for name, _ in MO.SHAPES:
        a, b = gd[name].reshape(-1), rd[name].reshape(-1)
        nb = np.linalg.norm(b)
        # a BF16 activation or pooled row on a rounding edge may fall either way: 2^-8 of a
        # row's share each, and with few candidates one row is a large share
        assert np.linalg.norm(a - b) <= 2e-2 * nb + 1e-12, (name, np.linalg.norm(a - b) / max(nb, 1e-30))
