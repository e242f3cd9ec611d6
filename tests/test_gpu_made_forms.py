"""The learned proposal's kernels on both sides of the sizes at which another
form takes over, through the C ABI, against numpy."""
import numpy as np
import pytest

from test_gpu_made import _to_bf16_bits
from test_gpu_made_kernels import _arrays

pytestmark = pytest.mark.gpu


# 128 x 128 tiles two to a CU: from K = 384 on, whole steps of 64 and not
@pytest.mark.parametrize("M,N,K", [(2056, 4104, 376), (2056, 4104, 384), (2904, 2952, 8), (2048, 4096, 456)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_tiles_by_depth(gpu_ok, M, N, K, ta, tb):
    """Small integers: every product and sum is exact."""
    from mi3gpu._lib import lib
    rng = np.random.default_rng(M + K)
    A = rng.integers(-4, 5, (M, K)).astype(np.float32)
    B = rng.integers(-4, 5, (K, N)).astype(np.float32)
    d = _arrays(A=_to_bf16_bits(A.T.copy() if ta else A), B=_to_bf16_bits(B.T.copy() if tb else B),
                C=np.zeros((M, N), 'f4'))
    assert lib().mi3_gemm_bf16(d.stream, ta, tb, M, N, K, 2.0, d['A'], M if ta else K, d['B'],
                               K if tb else N, 0.0, d['C'], N, None, 0, None, 0) == 0
    d.sync()
    np.testing.assert_array_equal(d.read('C'), 2 * (A @ B))
    d.close()


# one unit of a sequence to a thread; four of one (393216 units on) and of four (1572864);
# four sequences of a unit where units are no multiple of 4 (786432)
@pytest.mark.parametrize("L,q,H,B", [(9, 21, 512, 768), (9, 21, 512, 769), (6, 4, 512, 3072), (6, 4, 512, 3075), (5, 25, 4, 98305),
                                     (7, 3, 250, 3145), (7, 3, 250, 3147), (4, 17, 6, 131073), (300, 21, 64, 17)])
def test_embedding_by_size(gpu_ok, L, q, H, B):
    from mi3gpu._lib import lib
    rng = np.random.default_rng(B)
    ld = B + 5
    s = rng.integers(0, q, (L, ld)).astype('u1')
    W = rng.normal(size=(L * q, H)).astype('f4')
    b1 = rng.normal(size=H).astype('f4')
    d = _arrays(s=s, W=W, b1=b1, h=np.zeros((B, H), 'f4'), hb=np.zeros((B, H), 'u2'))
    assert lib().mi3_made_embed(d.stream, d['s'], ld, B, L, q, H, d['W'], d['b1'], d['h'], d['hb']) == 0
    d.sync()
    h = np.repeat(b1[None], B, axis=0)      # float32, sites in order, as the kernel adds
    for i in range(L):
        h += W[i * q + s[i, :B].astype(int)]
    np.testing.assert_array_equal(d.read('h'), h)
    np.testing.assert_array_equal(d.read('hb'), _to_bf16_bits(np.maximum(h, 0)))
    d.close()


def test_embedding_of_nothing_is_refused(gpu_ok):
    from mi3gpu._lib import lib
    d = _arrays(s=np.zeros((2, 16), 'u1'), W=np.zeros((8, 4), 'f4'), b=np.zeros(4, 'f4'), h=np.zeros(4, 'f4'))
    for B, H in ((0, 4), (4, 0)):
        assert lib().mi3_made_embed(d.stream, d['s'], 16, B, 2, 4, H, d['W'], d['b'], d['h'], d['h']) < 0
    d.close()


# up to 7 q sequences without a sort, more where there are many work-groups (the last
# two); groups of 64 and chunks of 2048 sorted
@pytest.mark.parametrize("L,q,H,B", [(5, 2, 1, 1), (7, 21, 260, 147), (7, 21, 260, 148), (7, 21, 257, 149), (3, 25, 256, 175),
                                     (3, 25, 66, 176), (9, 4, 512, 28), (9, 4, 512, 29), (4, 4, 64, 63), (4, 4, 64, 65),
                                     (4, 9, 300, 2047), (4, 9, 64, 2049), (200, 3, 515, 215), (200, 3, 515, 216)])
def test_embedding_gradient_by_size(gpu_ok, L, q, H, B):
    from mi3gpu._lib import lib
    rng = np.random.default_rng(B)
    ld = B + 5
    s = rng.integers(0, q, (L, ld)).astype('u1')
    dh = rng.normal(size=(B, H)).astype('f4')
    d = _arrays(s=s, dh=dh, dW=np.ones((L * q, H), 'f4'))
    assert lib().mi3_made_embed_grad(d.stream, d['s'], ld, B, L, q, H, d['dh'], d['dW']) == 0
    d.sync()
    dW = np.zeros((L * q, H), 'f4')      # float32, in batch order, as the kernels add
    for b in range(B):
        dW[np.arange(L) * q + s[:, b]] += dh[b]
    np.testing.assert_array_equal(d.read('dW'), dW)
    d.close()
