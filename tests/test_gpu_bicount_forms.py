"""Every form of the bicounts (three and five bit planes, both block sizes and
stage lengths, whole blocks and shared ones) against integer counts, exactly."""
import numpy as np
import pytest

from mi3gpu._lib import lib, check
from oracle import cboracle
from test_gpu_kernels import make_gpu, seqs_rand

pytestmark = pytest.mark.gpu

# (L, q, sequences): q at the edges of the planes and stages, L*q at the edges of
# blocks, sequences at the edges of units (128), stages (5 or 3 units) and parts
CASES = [(2, 2, 1), (3, 2, 127), (32, 2, 128), (33, 2, 129), (450, 2, 65601),
         (43, 3, 641), (64, 4, 384), (16, 7, 385), (147, 7, 65537), (150, 7, 4095),
         (16, 8, 640), (17, 8, 4097), (146, 8, 66001), (61, 16, 5000), (300, 21, 700),
         (255, 25, 4100), (51, 25, 16385), (3, 25, 2)]


def counts_of(tmp_path, L, q, s):
    g = make_gpu(tmp_path, L, q, 512, wgsize=512)
    g.initLargeBufs(len(s))
    g.setBuf('seq large', s)
    g.calcBicounts('large')
    return g, g.getBuf('bicount').read()


@pytest.mark.parametrize("L,q,n", CASES)
def test_bicount_forms(gpu_ok, tmp_path, L, q, n):
    s = seqs_rand(n, L, q, 7)
    s[:, -1] = q - 1
    np.testing.assert_array_equal(counts_of(tmp_path, L, q, s)[1], cboracle.bicounts(s, q))


def test_bicount_one_letter_past_a_float_sum(gpu_ok, tmp_path):
    """More sequences with the same letters than one float32 sum takes; then none."""
    L, q, n = 3, 2, 2 ** 23 + 77
    g, c = counts_of(tmp_path, L, q, np.ones((n, L), '<u1'))
    assert np.array_equal(c, np.tile(np.array([0, 0, 0, n], '<u4'), (3, 1)))
    check(g._ctx, lib().mi3_calc_bicounts(g._ctx, b'seq large', 0))
    assert not g.getBuf('bicount').read().any()
