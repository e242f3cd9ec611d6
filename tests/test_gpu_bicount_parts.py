"""Bicounts where a wave's sequences exceed what it sums at a time (2^23)."""
import numpy as np
import pytest

from mi3gpu._lib import lib, check
from oracle import cboracle
from test_gpu_kernels import seqs_rand

pytestmark = pytest.mark.gpu


# 32 parts of a single block; waves that take a block and a part of the next
@pytest.mark.parametrize("L,q,n", [(2, 2, 2 ** 28 + 32 * 11 * 128 + 77), (254, 25, 2 ** 23 + 5 * 128 + 3)])
def test_bicount_parts(gpu_ok, L, q, n):
    """One sequence throughout, but for some at each end."""
    import ctypes
    from mi3gpu._lib import as_ptr
    ld, m = (n + 15) // 16 * 16, 1000
    ctx = ctypes.c_void_p()
    check(None, lib().mi3_create(0, L, q, 512, 1, 0, ctypes.byref(ctx)))
    nb = L * (L - 1) // 2 * q * q
    try:
        check(ctx, lib().mi3_buf_alloc(ctx, b'seq large', L * ld))
        check(ctx, lib().mi3_buf_alloc(ctx, b'bicount', nb * 4))
        one = np.arange(L, dtype='u1') % q
        check(ctx, lib().mi3_fill_seqs(ctx, b'seq large', as_ptr(one)))
        ends = [seqs_rand(m, L, q, 1), seqs_rand(m, L, q, 2)]
        for e, at in zip(ends, (0, n - m)):
            for i in range(L):
                row = np.ascontiguousarray(e[:, i])
                check(ctx, lib().mi3_buf_write(ctx, b'seq large', as_ptr(row), m, i * ld + at))
        check(ctx, lib().mi3_calc_bicounts(ctx, b'seq large', n))
        got, t = np.empty(nb, '<u4'), ctypes.c_int()
        check(ctx, lib().mi3_buf_read_async(ctx, b'bicount', got.nbytes, 0, ctypes.byref(t)))
        check(ctx, lib().mi3_ticket_wait(ctx, t, as_ptr(got), got.nbytes))
    finally:
        lib().mi3_destroy(ctx)
    want = cboracle.bicounts(np.concatenate(ends), q).reshape(-1, q * q)
    i, j = np.triu_indices(L, 1)
    want[np.arange(len(i)), one[i].astype(int) * q + one[j]] += np.uint32(n - 2 * m)
    np.testing.assert_array_equal(got.reshape(-1, q * q), want)
