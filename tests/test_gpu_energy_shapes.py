"""Energies of staged rows on both sides of the counts at which their shape
changes, against the float64 oracle."""
import numpy as np
import pytest

from oracle import cboracle
from test_gpu_kernels import make_gpu, model, seqs_rand

pytestmark = pytest.mark.gpu


# 32768 to 65536 sequences of a 256-CU card: 16 waves of 8 slots for up to 4 chunks
@pytest.mark.parametrize("L,q,n", [(31, 5, 32769), (33, 8, 33000), (66, 6, 45987), (128, 7, 49155), (97, 8, 65536), (97, 8, 65537),
                                   (129, 8, 40001)])
def test_energy_shapes(gpu_ok, tmp_path, L, q, n):
    J = model(L, q, 3)
    s = seqs_rand(n, L, q, 4)
    g = make_gpu(tmp_path, L, q, 512, wgsize=512)
    g.initLargeBufs(n)
    g.setBuf('J', J)
    g.setBuf('seq large', s)
    g.calcEnergies('large')
    E = g.getBuf('E large').read()
    # float32 sums of L(L-1)/2 terms: 1e-5 of the sum of magnitudes, as for the other sizes
    assert (np.abs(E - cboracle.energies(s, J)) / cboracle.energies(s, np.abs(J))).max() < 1e-5
