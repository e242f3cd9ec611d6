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


# state words of one to five and more, chunks of each class
STAGED = [[(20, 4, 20480), (17, 2, 512)], [(24, 21, 17408), (33, 17, 1024)], [(131, 9, 18432)], [(260, 3, 16896)],
          [(24, 12, 8704), (12, 16, 512)], [(390, 17, 1024)], [(520, 4, 8704)]]


@pytest.mark.parametrize("models", STAGED)
@pytest.mark.parametrize("tile", [None, 128, 256, 512])
def test_batch_staged_tiles(gpu_ok, models, tile):
    """Tiles asked for by size, and, for classes of many walkers, the library's choice."""
    b, data = _batch(models, tile)
    b.run(1)
    b.run(1)
    for m, (L, q, N) in enumerate(models):
        _check_model(b.get_seqs(m), data[m][1], data[m][0], 40 + m, [(0, L), (L + (L & 1), L)])
        assert b.tile(m) == min(tile or 512, 256 if L > 512 else 512)
    b.close()


# 2049 to 8192 walkers of more than 8 letters (four to a half-wave), one model or
# several, state words of one to five; and one to a half-wave
UNSTAGED = [[(40, 21, 1536), (33, 17, 1536), (37, 21, 512)], [(140, 9, 2560), (129, 16, 1024)], [(260, 12, 2560)],
            [(390, 21, 2560)], [(520, 9, 2560)], [(30, 25, 1024), (21, 22, 2048)], [(50, 4, 3584), (64, 8, 512)]]


@pytest.mark.parametrize("models", UNSTAGED)
def test_batch_unstaged(gpu_ok, models):
    b, data = _batch(models)
    b.run(1)
    b.run(1)
    for m, (L, q, N) in enumerate(models):
        _check_model(b.get_seqs(m), data[m][1], data[m][0], 40 + m, [(0, L), (L + (L & 1), L)])
    b.close()


# classes that are swept unstaged alone and staged together, and some of each
MIXED = [[(20, 21, 8192), (130, 21, 8192), (258, 21, 8192)], [(24, 21, 8192), (22, 25, 8192), (20, 16, 512), (33, 4, 6144)],
         [(20, 21, 2048), (130, 21, 8192), (258, 4, 8192), (300, 21, 1024)]]


@pytest.mark.parametrize("models", MIXED)
@pytest.mark.parametrize("tune", [False, True])
def test_batch_of_several_classes(gpu_ok, models, tune):
    b, data = _batch(models)
    if tune:
        b.tune(1)
        for m, (J, s0) in enumerate(data):
            b.set_seqs(m, s0)
    start = [b.step_count(m) for m in range(len(models))]
    b.run(1)
    b.run(1)
    for m, (L, q, N) in enumerate(models):
        t = start[m]
        _check_model(b.get_seqs(m), data[m][1], data[m][0], 40 + m, [(t, L), (t + L + (L & 1), L)])
        assert b.tile(m) in (128, 256, 512)
    b.close()
