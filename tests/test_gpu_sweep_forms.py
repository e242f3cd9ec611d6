"""Every form and tile that the sweep chooses by walker count (unstaged,
steps staged, chunks staged) gives the oracle's chains, and the same bytes as
a tile asked for by size."""
import numpy as np
import pytest

from oracle import cboracle
from test_gpu_kernels import make_gpu, model, seqs_rand

pytestmark = pytest.mark.gpu

# (L, q, walkers, steps): lengths at the edges of chunks (32), state words
# (128) and staged rows; walker counts at the edges of the forms and tiles of a
# 256-CU card
CASES = [(2, 2, 512, 7), (32, 4, 512, 41), (33, 25, 1024, 33), (129, 3, 3072, 20), (160, 21, 1536, 17),
         (97, 9, 1024, 12), (1024, 4, 512, 9),                      # unstaged
         (160, 21, 2048, 17), (31, 2, 3584, 65), (93, 8, 8192, 30), (93, 8, 8704, 30), (256, 6, 16384, 9), (385, 4, 6656, 11),
         (33, 4, 16896, 37), (225, 8, 66048, 6), (128, 7, 66048, 9), (300, 3, 66048, 5),
         (1000, 4, 16896, 5),                                       # steps staged
         (65, 9, 8704, 21), (300, 5, 8704, 9), (40, 21, 66048, 12), (70, 16, 131584, 6),
         (420, 21, 66048, 3), (600, 22, 16896, 4)]                  # chunks staged


@pytest.mark.parametrize("L,q,N,nsteps", CASES)
def test_sweep_forms(gpu_ok, tmp_path, L, q, N, nsteps):
    J = model(L, q, 7, sj=0.3 if q < 10 else 0.1)
    s0 = seqs_rand(N, L, q, 8)
    got = []
    for wg in (512, 128):
        g = make_gpu(tmp_path, L, q, N, seed=99, nsteps=nsteps, wgsize=wg)
        g.setBuf('J', J)
        g.setBuf('seq main', s0)
        g.runMCMC()
        g.runMCMC()
        got.append(g.getBuf('seq main').read())
        del g
    np.testing.assert_array_equal(got[0], got[1])
    want, m1 = cboracle.metropolis(s0, J, 99, 0, nsteps)
    want, m2 = cboracle.metropolis(want, J, 99, nsteps + (nsteps & 1), nsteps)
    same = np.all(got[0] == want, axis=1)
    assert np.all(same[np.minimum(m1, m2) > 1e-3])
    assert same.mean() > 0.98
