"""Every form and tile that the energies choose by sequence count (unstaged,
rows staged, chunks staged) against the float64 oracle, on ragged sets."""
import numpy as np
import pytest

from oracle import cboracle
from test_gpu_kernels import make_gpu, model, seqs_rand

pytestmark = pytest.mark.gpu

# (L, q, sequences): lengths at the edges of chunks (32), state words (128) and
# staged rows; counts at the edges of the forms and tiles of a 256-CU card
CASES = [(2, 2, 1), (32, 4, 33), (33, 25, 2047), (129, 21, 2048), (97, 7, 4096), (1024, 3, 600),   # unstaged
         (31, 2, 4097), (93, 8, 8191), (93, 8, 16385), (256, 6, 13001), (256, 8, 66001), (385, 4, 12301), (64, 5, 70003),
         (300, 3, 66003), (1000, 4, 14001),                                                         # rows staged
         (33, 9, 2049), (128, 16, 140001), (129, 21, 33333), (300, 5, 70001), (400, 21, 9001),
         (450, 17, 66001), (600, 22, 6001)]                                                         # chunks staged


@pytest.mark.parametrize("L,q,n", CASES)
def test_energy_forms(gpu_ok, tmp_path, L, q, n):
    J = model(L, q, 3)
    s = seqs_rand(n, L, q, 4)
    g = make_gpu(tmp_path, L, q, 512, wgsize=512)
    g.initLargeBufs(n)
    g.setBuf('J', J)
    g.setBuf('seq large', s)
    g.calcEnergies('large')
    E = g.getBuf('E large').read()
    # float32 sums of L(L-1)/2 terms: 1e-5 of the sum of magnitudes, as for the other sizes
    err = np.abs(E - cboracle.energies(s, J)) / cboracle.energies(s, np.abs(J))
    assert E.shape == (n,) and err.max() < 1e-5


# (L, q, sequences): folded sites that end with the chain and past it, one and two
# chunks of them, counts on both sides of the rule
@pytest.mark.parametrize("L,q,n", [(32, 2, 65537), (97, 2, 66000), (98, 2, 65552), (33, 3, 65537), (64, 4, 65536),
                                   (65, 4, 65537), (130, 4, 65553), (32, 5, 70001), (67, 5, 65537)])
def test_energies_folded(gpu_ok, tmp_path, L, q, n):
    """Also after the couplings change, and (folded: the other forms turn an infinite
    coupling into NaN) with forbidden pairs of letters, whose energies alone are
    infinite."""
    s = seqs_rand(n, L, q, 4)
    g = make_gpu(tmp_path, L, q, 512, wgsize=512)
    g.initLargeBufs(n)
    g.setBuf('seq large', s)
    for seed in (3, 4):
        J = model(L, q, seed)
        want, mag = cboracle.energies(s, J), cboracle.energies(s, np.abs(J))
        forbid = seed == 4 and n > 65536
        if forbid:   # sites 0 and 1, letters 1 and 0; the last two sites, 0 and 1
            J[0, q] = J[-1, 1] = np.inf
        g.setBuf('J', J)
        g.calcEnergies('large')
        E = g.getBuf('E large').read()
        no = (((s[:, 0] == 1) & (s[:, 1] == 0)) | ((s[:, -2] == 0) & (s[:, -1] == 1))) & forbid
        assert np.array_equal(np.isposinf(E), no)
        assert (np.abs(E - want) / mag)[~no].max() < 1e-5
