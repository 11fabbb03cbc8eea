"""GPU tests of the Hausdorff query's pruning: sample counts around its batches, tiny targets, repeated maxima."""
import numpy as np
import pytest

import oracle
from cuacd_amd import datasets

pytestmark = pytest.mark.gpu


def _pairs():
    ico = datasets.noisy_icospheres(1, 3, 0.2, seed=5)[0]
    box = datasets.box_mesh((-1, -1, -1), (1, 1, 1))
    tri = (np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0]], np.float32), np.array([[0, 1, 2]], np.int32))
    far = (ico[0] + np.float32(50.0), ico[1])
    return [(ico, box), (box, ico), (ico, tri), (tri, ico), (ico, ico), (ico, far), (box, box)]


@pytest.mark.parametrize("n", [1, 63, 255, 256, 257, 511, 513, 1023, 1024, 1025, 3000])
def test_stratified_distances_match_brute_force(ctx, n):
    a, b = [p[0] for p in _pairs()], [p[1] for p in _pairs()]
    ab, ba, sa, sb = ctx.batch_hausdorff(a, b, n_samples=n, return_samples=True)
    for i in range(len(a)):
        # FP32 point-triangle distances of coordinates up to c round to about
        # 4 ulp of c: 4 * 2^-23 * 53 = 2.5e-5 for the pair 50 apart, whose
        # squared distance rounds relatively
        tol = 2.5e-5 if i == 5 else 1e-5
        assert abs(ab[i] - oracle.directed_hausdorff(sa[i], *b[i])) <= tol, i
        assert abs(ba[i] - oracle.directed_hausdorff(sb[i], *a[i])) <= tol, i


@pytest.mark.parametrize("copies", [1, 20])
def test_reference_sampler_is_the_same_alone_and_in_a_batch(ctx, copies):
    """The share of samples per workgroup depends on the batch; the distances do not."""
    p = _pairs()
    ab, ba = ctx.batch_hausdorff([x for x, _ in p] * copies, [y for _, y in p] * copies, sampler="reference")
    for i, (x, y) in enumerate(p):
        one = ctx.batch_hausdorff([x], [y], sampler="reference")
        for k in range(copies):
            got, want = (ab[i + k * len(p)], ba[i + k * len(p)]), (one[0][0], one[1][0])
            # the nearest triangle is the same up to the rounding of two squared distances
            assert np.allclose(got, want, rtol=2e-6, atol=0)


@pytest.mark.parametrize("copies", [1, 24])
def test_running_maximum_shared_by_waves_gives_the_same_bits(ctx, copies):
    """Waves raise the maximum while others search against it: no interleaving may lose a distance or change one."""
    p = _pairs() + [tuple(datasets.noisy_icospheres(2, 3, 0.1, seed=7))]
    n = 3000  # several batches of samples per workgroup and several workgroups per pair
    want = None
    for _ in range(6):
        ab, ba = ctx.batch_hausdorff([x for x, _ in p] * copies, [y for _, y in p] * copies, n_samples=n)
        got = np.stack([ab, ba]).reshape(2, copies, len(p))
        want = got[:, :1] if want is None else want
        assert np.array_equal(got, np.broadcast_to(want, got.shape))
