"""Weighted marginals of reduced alphabets, counted over folded sites, exactly."""
import numpy as np
import pytest

from test_gpu_kernels import make_gpu, seqs_rand

pytestmark = pytest.mark.gpu


# (L, q, sequences): folded sites that end with the chain and past it, counts on both
# sides of the rule and ragged
@pytest.mark.parametrize("L,q,n", [(47, 2, 65537), (48, 2, 65568), (49, 2, 66001), (33, 2, 65537), (53, 3, 66001),
                                   (54, 3, 65555), (93, 4, 65999), (94, 4, 65537), (94, 4, 65536), (143, 5, 65553),
                                   (144, 5, 70016)])
def test_weighted_marginals_folded(gpu_ok, tmp_path, L, q, n):
    """Whole weights whose sum is a power of two: every step is exact."""
    rng = np.random.default_rng(L + q)
    s = seqs_rand(n, L, q, 4)
    w = rng.integers(0, 8, n)
    w[0] += 2 ** 19 - w.sum()
    assert w[0] >= 0
    g = make_gpu(tmp_path, L, q, 512, wgsize=512)
    g.initLargeBufs(n)
    g.setBuf('seq large', s)
    g.initJstep()
    g.setBuf('weights large', w.astype('<f4'))
    g.weightedMarg('large')
    X = (s[:, :, None] == np.arange(q)).reshape(n, L * q).astype(np.float64)
    want = ((X.T * w) @ X).reshape(L, q, L, q).transpose(0, 2, 1, 3).reshape(L, L, q * q)
    np.testing.assert_array_equal(g.getBuf('bi').read(), want[np.triu_indices(L, 1)])
