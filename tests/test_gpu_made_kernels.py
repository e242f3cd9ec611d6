"""The learned proposal's training kernels at the edges of their tiles, through
the C ABI, against numpy in float64."""
import numpy as np
import pytest

from test_gpu_made import _from_bf16_bits, _to_bf16_bits

pytestmark = pytest.mark.gpu


def _arrays(**kw):
    from mi3gpu.made import DeviceArrays
    d = DeviceArrays()
    for k, v in kw.items():
        d.alloc(k, v.shape, v.dtype)
        d.write(k, v)
    return d


# one piece; both sides of a 64-tile and a K step; enough 128-tiles to be taken
@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (64, 64, 64), (72, 136, 200), (56, 248, 72), (4104, 2056, 72)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_tile_edges(gpu_ok, M, N, K, ta, tb):
    """Small integers: every product and sum is exact."""
    from mi3gpu._lib import lib
    rng = np.random.default_rng(M + K)
    A = rng.integers(-4, 5, (M, K)).astype(np.float32)
    B = rng.integers(-4, 5, (K, N)).astype(np.float32)
    d = _arrays(A=_to_bf16_bits(A.T.copy() if ta else A), B=_to_bf16_bits(B.T.copy() if tb else B),
                C=np.zeros((M, N), 'f4'), Cb=np.zeros((M, N), 'u2'))
    assert lib().mi3_gemm_bf16(d.stream, ta, tb, M, N, K, 2.0, d['A'], M if ta else K, d['B'],
                               K if tb else N, 0.0, d['C'], N, d['Cb'], N, None, 0) == 0
    d.sync()
    np.testing.assert_array_equal(d.read('C'), 2 * (A @ B))
    d.close()


# (L, q, B, H): vector and scalar forms, batches that end inside a group of 4
# sequences, 64 or 2048 letters, more than 256 sites, odd numbers of sites
@pytest.mark.parametrize("L,q,B,H", [(2, 2, 1, 1), (5, 3, 7, 30), (16, 21, 64, 64), (33, 25, 70, 68),
                                     (257, 4, 300, 32), (300, 7, 33, 130),
                                     (3, 20, 2050, 260)])
def test_embedding_and_softmax(gpu_ok, L, q, B, H):
    from mi3gpu._lib import lib
    rng = np.random.default_rng(L)
    ld = B + 3
    s = rng.integers(0, q, (L, ld)).astype('u1')
    W = rng.normal(size=(L * q, H)).astype('f4')
    b1 = rng.normal(size=H).astype('f4')
    dh = rng.normal(size=(B, H)).astype('f4')
    z = rng.normal(0, 2, size=(B, L * q)).astype('f4')
    d = _arrays(s=s, W=W, b1=b1, dh=dh, z=z, h=np.zeros((B, H), 'f4'), hb=np.zeros((B, H), 'u2'),
                dW=np.zeros((L * q, H), 'f4'), nll=np.zeros(B, 'f4'), g=np.zeros((B, L * q), 'f4'),
                gb=np.zeros((B, L * q), 'u2'))
    l = lib()
    assert l.mi3_made_embed(d.stream, d['s'], ld, B, L, q, H, d['W'], d['b1'], d['h'], d['hb']) == 0
    assert l.mi3_made_embed_grad(d.stream, d['s'], ld, B, L, q, H, d['dh'], d['dW']) == 0
    assert l.mi3_made_xent(d.stream, d['z'], d['s'], ld, B, L, q, 0.5, d['nll'], d['gb'], d['g']) == 0
    d.sync()
    idx = np.arange(L)[:, None] * q + s[:, :B]                      # (L, B)
    # float32 sums of L (B) terms of size 1: a few units in the last place of each
    h = b1 + W.astype('f8')[idx].sum(axis=0)
    np.testing.assert_allclose(d.read('h'), h, rtol=0, atol=2e-6 * L + 1e-6)
    assert np.abs(_from_bf16_bits(d.read('hb')) - np.maximum(h, 0)).max() <= np.abs(h).max() / 128
    dW = np.zeros((L * q, H))
    for i in range(L):
        np.add.at(dW, idx[i], dh)
    np.testing.assert_allclose(d.read('dW'), dW, rtol=0, atol=2e-6 * B + 1e-6)
    zz = z.astype('f8').reshape(B, L, q)
    lse = np.log(np.exp(zz).sum(axis=2))
    hot = np.arange(q)[None, None, :] == s[:, :B].T[:, :, None]
    np.testing.assert_allclose(d.read('nll'), (lse - zz[hot].reshape(B, L)).sum(axis=1), rtol=0,
                               atol=5e-6 * L + 1e-6)
    g = 0.5 * (np.exp(zz - lse[:, :, None]) - hot).reshape(B, -1)
    np.testing.assert_allclose(d.read('g'), g, rtol=0, atol=2e-6)
    np.testing.assert_allclose(_from_bf16_bits(d.read('gb')), g, rtol=0, atol=0.5 / 128)
    d.close()


# one row, one column, either side of the 8 row lanes and of their 32 loads
@pytest.mark.parametrize("rows,cols", [(1, 1), (7, 33), (249, 31), (256, 64), (4096, 512), (1000, 4872)])
def test_column_sums(gpu_ok, rows, cols):
    from mi3gpu._lib import lib
    x = np.random.default_rng(cols).normal(size=(rows, cols)).astype('f4')
    d = _arrays(x=x, o=np.zeros(cols, 'f4'))
    assert lib().mi3_colsum(d.stream, rows, cols, d['x'], d['o']) == 0
    d.sync()
    np.testing.assert_allclose(d.read('o'), x.astype('f8').sum(axis=0), rtol=0, atol=2e-6 * rows)
    d.close()


# (L, q, H, B): each number of k-steps per wave (H to 128, 256, 384, 512) full and
# ragged, one and two column tiles of letters, more than 16 units of a degree and
# fewer units than degrees, walkers that end inside a tile
@pytest.mark.parametrize("L,q,H,B", [(2, 4, 32, 1), (8, 17, 128, 33), (40, 25, 160, 64), (24, 2, 256, 16),
                                     (56, 21, 288, 100), (16, 10, 384, 1000), (600, 4, 416, 20),
                                     (4, 16, 512, 17), (24, 21, 480, 50)])
def test_fused_draws(gpu_ok, L, q, H, B):
    from mi3gpu.made import MADE
    from oracle import made_oracle as mo
    from oracle.philox import philox4x32_10
    from test_gpu_made import _params, _perturb
    from mi3gpu._lib import lib
    m = MADE(L, q, H, max_batch=16, seed=4)
    _perturb(m, np.random.default_rng(8), {'W1t': 0.1, 'b1': 0.1, 'W2': 0.1, 'b2': 0.1, 'W3': 0.1, 'b3': 0.5})
    ld = (B + 15) // 16 * 16
    m.mem.alloc('out', (L, ld), 'u1')
    m.mem.alloc('drawn', (B,), 'f4')
    m.mem.alloc('read', (B,), 'f4')
    for nll, draw in (('drawn', 1), ('read', 0)):
        assert lib().mi3_made_fused(m.mem.stream, L, q, H, B, *[m.mem[k] for k in ('W1t', 'b1', 'W2b', 'b2', 'W3b', 'b3')],
                                    5 + (7 << 32), 9, 3, m.mem['out'], ld, m.mem[nll], draw) == 0
    s = m.get('out').T[:B]
    np.testing.assert_array_equal(m.get('drawn'), m.get('read'))
    # a unit that rounds to the other bfloat16 neighbour (2^-8 of a value of at most
    # 2) moves a logit by up to 2e-3; two of them are allowed for
    f = mo.forward(s, *_params(m), q, bf=True)
    np.testing.assert_allclose(m.get('read'), f['nll'], rtol=1e-4, atol=5e-3)
    z = f['logits'].reshape(B, L, q)
    cdf = np.cumsum(np.exp(z - f['lse'][..., None]), axis=2)
    j, b = np.meshgrid(np.arange(L, dtype=np.uint32), 3 + np.arange(B, dtype=np.uint32))
    one = np.ones_like(j)
    u = (philox4x32_10(j, b, 9 * one, 0x4D414445 * one, 5, 7)[0] >> 8) * 2.0 ** -24
    want = np.minimum((cdf <= u[..., None]).sum(axis=2), q - 1)
    clear = np.abs(cdf - u[..., None]).min(axis=2) > 5e-3
    assert clear.mean() > 0.5 and np.array_equal(want[clear], s[clear])
    m.close()
