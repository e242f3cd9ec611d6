"""Sequences and couplings at the edges of what the engine accepts, and its
calls under graph capture."""
import ctypes

import numpy as np
import pytest

from mi3gpu._lib import lib, check
from test_gpu_kernels import make_gpu, model, seqs_rand

pytestmark = pytest.mark.gpu


def _write(g, name, a):
    check(g._ctx, lib().mi3_buf_write(g._ctx, name, a.ctypes.data, a.nbytes, 0))


@pytest.mark.parametrize("L,q,n", [(40, 4, 300), (65, 21, 515), (130, 9, 77)])
def test_unstaged_energies_of_forbidden_pairs(gpu_ok, tmp_path, L, q, n):
    """An infinite coupling makes the energies of the sequences that hold it infinite and no others:
    pairs within a chunk of 32 sites, its last site, across chunks, and the last sites."""
    J = model(L, q, 3)
    s = seqs_rand(n, L, q, 4)
    hold = np.zeros(n, bool)
    for i, j in ((0, 1), (3, 31), (5, 20), (30, 31), (31, 32), (2, L - 2), (L - 3, L - 1), (L - 2, L - 1)):
        J[i * (2 * L - i - 1) // 2 + j - i - 1, 1 * q + 2] = np.inf
        hold |= (s[:, i] == 1) & (s[:, j] == 2)
    assert hold.any() and not hold.all()
    g = make_gpu(tmp_path, L, q, 512, wgsize=512)
    g.initLargeBufs(n)
    g.setBuf('J', J)
    g.setBuf('seq large', s)
    g.calcEnergies('large')
    E = g.getBuf('E large').read()
    np.testing.assert_array_equal(np.isposinf(E), hold)
    assert np.isfinite(E[~hold]).all()


@pytest.mark.parametrize("L,q,n", [(5, 2, 129), (40, 4, 1000), (7, 7, 640), (9, 8, 640), (6, 25, 300)])
def test_bicounts_bytes_that_are_no_letter(gpu_ok, tmp_path, L, q, n):
    rng = np.random.default_rng(q)
    s = seqs_rand(n, L, q, 5)
    odd = rng.random(s.shape) < 0.3
    s[odd] = rng.choice([q, 7, 8, 9, 31, 32, 33, 64, 127], size=odd.sum())
    g = make_gpu(tmp_path, L, q, 512, wgsize=512)
    g.initLargeBufs(n)
    dev = np.zeros((L, g._seq_ld('seq large')), 'u1')
    dev[:, :n] = s.T
    _write(g, b'seq large', dev)
    check(g._ctx, lib().mi3_calc_bicounts(g._ctx, b'seq large', n))
    X = (s[:, :, None] == np.arange(q)).reshape(n, L * q).astype(np.int64)
    want = (X.T @ X).reshape(L, q, L, q).transpose(0, 2, 1, 3).reshape(L, L, q * q)
    np.testing.assert_array_equal(g.getBuf('bicount').read(), want[np.triu_indices(L, 1)])


def test_a_byte_that_is_no_letter_stays_in_its_sequence(gpu_ok, tmp_path):
    """q = 16: the letter 16 (at rows within the staged couplings) changes no other
    sequence's energy and no other walker's chain."""
    L, q, N = 40, 16, 2560
    J = model(L, q, 3)
    s = seqs_rand(N, L, q - 2, 4)
    at = np.arange(0, N, 7)
    res = []
    for letter in (0, q):
        g = make_gpu(tmp_path, L, q, N, seed=9, nsteps=L, wgsize=512)
        dev = np.ascontiguousarray(s.T)
        dev[3, at] = letter
        g.setBuf('J', J)
        _write(g, b'seq main', dev)
        g.calcEnergies('main')
        E = g.getBuf('E main').read()
        g.runMCMC()
        out = np.empty_like(dev)
        t = ctypes.c_int()
        check(g._ctx, lib().mi3_buf_read_async(g._ctx, b'seq main', out.nbytes, 0, ctypes.byref(t)))
        check(g._ctx, lib().mi3_ticket_wait(g._ctx, t, out.ctypes.data, out.nbytes))
        rest = np.setdiff1d(np.arange(N), at)
        res.append((E[rest], out[:, rest]))
    np.testing.assert_array_equal(res[0][0], res[1][0])
    np.testing.assert_array_equal(res[0][1], res[1][1])


class _Graph:
    """What a block of calls enqueues on a context's stream, captured."""

    def __init__(self, g):
        self.s = ctypes.c_void_p()
        check(g._ctx, lib().mi3_stream(g._ctx, ctypes.byref(self.s)))

    def _hip(self, name, *a):
        f = getattr(lib(), name)      # from the HIP runtime that the library is linked to
        f.restype = ctypes.c_int
        assert f(*a) == 0, name

    def __enter__(self):
        self._hip('hipStreamBeginCapture', self.s, 1)
        return self

    def __exit__(self, *exc):
        self.graph, self.exec = ctypes.c_void_p(), ctypes.c_void_p()
        f = lib().hipStreamEndCapture
        f.restype = ctypes.c_int
        rc = f(self.s, ctypes.byref(self.graph))
        if exc[0] is None:
            assert rc == 0
            self._hip('hipGraphInstantiate', ctypes.byref(self.exec), self.graph, None, None, ctypes.c_size_t(0))

    def launch(self):
        self._hip('hipGraphLaunch', self.exec, self.s)

    def close(self):
        self._hip('hipGraphExecDestroy', self.exec)
        self._hip('hipGraphDestroy', self.graph)


@pytest.mark.parametrize("L,q", [(30, 4), (40, 21)])
def test_bicounts_captured(gpu_ok, tmp_path, L, q):
    """The context's first count is captured; replays stay right when larger sets are counted between."""
    from oracle import cboracle
    N, n = 1024, 9000
    a, b = seqs_rand(N, L, q, 1), seqs_rand(n, L, q, 2)
    g = make_gpu(tmp_path, L, q, N)
    g.initLargeBufs(n)
    g.setBuf('seq main', a)
    g.setBuf('seq large', b)
    with _Graph(g) as cap:
        g.calcBicounts('main')
    wa, wb = cboracle.bicounts(a, q), cboracle.bicounts(b, q)
    for k in range(3):
        cap.launch()
        np.testing.assert_array_equal(g.getBuf('bicount').read(), wa)
        g.calcBicounts('large')
        g.wait()
        np.testing.assert_array_equal(g.getBuf('bicount').read(), wb)
    cap.close()
