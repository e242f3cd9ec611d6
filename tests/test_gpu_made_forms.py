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
