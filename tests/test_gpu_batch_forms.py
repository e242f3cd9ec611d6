"""Every form that a batch sweeps its classes in gives the single-model chains."""
import numpy as np
import pytest

from test_gpu_batch import _check_model

pytestmark = pytest.mark.gpu


def _batch(models, tile=None):
    from mi3gpu.batch import PottsBatch
    L, q, N = zip(*models)
    b = PottsBatch(L, q, N, seed=40)
    data = []
    for m, (Lm, qm, Nm) in enumerate(models):
        rng = np.random.default_rng(200 + m)
        J = rng.normal(0, 0.3 if qm < 10 else 0.1, size=(Lm * (Lm - 1) // 2, qm * qm)).astype('<f4')
        s0 = rng.integers(0, qm, size=(Nm, Lm)).astype('u1')
        b.set_couplings(m, J)
        b.set_seqs(m, s0)
        if tile:
            b.set_tile(m, min(tile, 256) if Lm > 512 else tile)
        data.append((J, s0))
    return b, data


# (L, q, walkers): more letters than leave room beside two chunks in the LDS
@pytest.mark.parametrize("tile", [None, 128, 256, 512])
def test_batch_of_the_largest_alphabets(gpu_ok, tile):
    models = [(22, 25, 8704), (30, 22, 512)]
    b, data = _batch(models, tile)
    b.run(1)
    b.run(1)
    for m, (L, q, N) in enumerate(models):
        _check_model(b.get_seqs(m), data[m][1], data[m][0], 40 + m, [(0, L), (L + (L & 1), L)])
    b.close()
