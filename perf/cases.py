"""The work that a user of this engine has it do, at the sizes that its bench, tests and command line use.

Each case goes through the package's own interface (MCMCGPU, GPU_node, NewtonSteps.iterNewton, PottsBatch, MADE, MixedSampler).
Sequences are drawn from skewed independent sites, as a run starts from; couplings hold the sites' fields plus weak random
pair terms, as an inference meets them.  Outputs are the engine's own device buffers, seen as tensors; the calls that hand
back host arrays (iterNewton, PottsBatch.get_seqs) return those.

`op` of a case:
  sweep     runMCMC: `nsteps` Metropolis site updates of N walkers
  measure   calcBicounts + bicounts_to_bimarg + calcEnergies of the walkers, as after every equilibration
  bicounts  bimarginals of a ragged set of stored sequences (the large buffer)
  energies  energies of a ragged set of stored sequences
  newton    quasi-Newton iterations on the engine's buffers (update, l1z, energies under dJ, weights, weighted marginals)
  iterate   a whole NewtonSteps.iterNewton call
  batch     models of uneven L and q swept together
  train     one MADE training step (loss, gradients, Adam)
  propose   one learned-proposal Metropolis-Hastings step of every walker
"""
import ctypes
import os
import sys
import tempfile
from pathlib import Path
from types import SimpleNamespace

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'mi3-gpu_amd'))

from mi3gpu._lib import lib, check  # noqa: E402
from mi3gpu.batch import PottsBatch  # noqa: E402
from mi3gpu.made import MADE, MixedSampler, made_masks, PARAMS  # noqa: E402
from mi3gpu.mcmcGPU import MCMCGPU  # noqa: E402
from mi3gpu.node_manager import GPU_node  # noqa: E402
from mi3gpu.NewtonSteps import iterNewton  # noqa: E402

WGSIZE = 512          # the command line's default work-group size
GAMMA, PC, LAM = 4e-4, 0.01, 1e-4   # step size, pc-damping and l1z strength of the HIV example
DEV = 'cuda:0'


def listed():
    return [
        # the smallest call: a few dozen site updates of one tile of walkers
        {'name': 'sweep_tiny', 'op': 'sweep', 'L': 40, 'q': 21, 'N': 512, 'nsteps': 80},
        # a CPU-sized problem moved to the GPU: 16384 walkers, 8 sweeps
        {'name': 'sweep_small', 'op': 'sweep', 'L': 99, 'q': 4, 'N': 16384, 'nsteps': 792},
        # the HIV protease example's launch
        {'name': 'sweep_hiv', 'op': 'sweep', 'L': 93, 'q': 4, 'N': 262144, 'nsteps': 2048},
        # the protein model of the bench: 8 sweeps of 2^18 walkers
        {'name': 'sweep_protein', 'op': 'sweep', 'L': 232, 'q': 21, 'N': 262144, 'nsteps': 1856},
        # eight small models of uneven length and alphabet in one graph
        {'name': 'batch_uneven', 'op': 'batch', 'nsweeps': 4,
         'models': '50x21x2048,57x4x1024,93x4x4096,111x21x1536,150x4x2048,232x21x2048,301x4x1024,400x21x1024'},
        # marginals and energies of the walkers of a small run
        {'name': 'measure_small', 'op': 'measure', 'L': 99, 'q': 4, 'N': 16384},
        # bimarginals of a long sampled alignment
        {'name': 'bicounts_large', 'op': 'bicounts', 'L': 232, 'q': 21, 'N': 1000003},
        # energies of a long protein's alignment
        {'name': 'energies_long', 'op': 'energies', 'L': 400, 'q': 21, 'N': 50001},
        # the quasi-Newton phase of the HIV example, as the driver calls it
        {'name': 'iterate_hiv', 'op': 'iterate', 'L': 93, 'q': 4, 'N': 262144, 'steps': 8},
        # quasi-Newton iterations of the protein model
        {'name': 'newton_protein', 'op': 'newton', 'L': 232, 'q': 21, 'N': 262144, 'steps': 2},
        # a training step of the learned proposal at the bench's size
        {'name': 'train_protein', 'op': 'train', 'L': 232, 'q': 21, 'H': 512, 'N': 4096},
        # a proposal step of every walker at the bench's size
        {'name': 'propose_protein', 'op': 'propose', 'L': 232, 'q': 21, 'H': 512, 'N': 65536},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case: any operation, sizes spread over their range, alphabets of nucleotides, reduced classes and residues."""
    op = rng.choice(['sweep', 'sweep', 'sweep', 'measure', 'bicounts', 'energies', 'newton', 'newton', 'iterate', 'batch',
                     'train', 'propose'])
    q = rng.choice([4, 21, rng.randint(2, 25)])
    L = _log_int(rng, 10, 450)
    if op == 'batch':
        models = []
        for _ in range(rng.randint(2, 8)):
            models.append('%dx%dx%d' % (_log_int(rng, 20, 400), rng.choice([4, 21, rng.randint(2, 25)]), 512 * rng.randint(1, 6)))
        return {'op': op, 'nsweeps': rng.randint(1, 4), 'models': ','.join(models)}
    if op in ('train', 'propose'):
        L = 8 * max(2, min(29, L // 8))
        H = 32 * rng.randint(2, 16)
        N = 512 * _log_int(rng, 1, 8) if op == 'train' else 512 * _log_int(rng, 1, 64)
        return {'op': op, 'L': L, 'q': q, 'H': H, 'N': N}
    if op in ('bicounts', 'energies'):
        # sequences of an alignment: any number of them
        top = min(500000, int(2.5e10 / (L * q) ** 2 * 400)) if op == 'bicounts' else min(400000, int(1.2e10 / L ** 2))
        return {'op': op, 'L': L, 'q': q, 'N': _log_int(rng, 1000, max(2000, top))}
    top = int(1.3e10 / (512 * L ** 2))
    N = 512 * _log_int(rng, 1, max(2, min(512, top)))
    if op == 'sweep':
        nsteps = max(16, min(int(L * rng.uniform(0.5, 8)), int(2.0e11 / (N * L))))
        return {'op': op, 'L': L, 'q': q, 'N': N, 'nsteps': nsteps}
    if op == 'measure':
        return {'op': op, 'L': L, 'q': q, 'N': N}
    if op == 'iterate':
        # whole calls move their arrays to the host: short chains and reduced alphabets
        return {'op': op, 'L': _log_int(rng, 10, 120), 'q': rng.choice([4, rng.randint(2, 8)]),
                'N': 512 * _log_int(rng, 1, 512), 'steps': rng.randint(2, 10)}
    return {'op': op, 'L': L, 'q': q, 'N': N, 'steps': 2}


def work(case):
    """Inputs read once and outputs written once; a site update, an energy and a marginal each take one term per partner."""
    op = case['op']
    if op == 'batch':
        b = f = 0.0
        for L, q, N in _models(case):
            b += 2.0 * N * L + 4.0 * _npairs(L) * q * q
            f += 2.0 * (L - 1) * N * L * case['nsweeps']
        return {'bytes': b, 'flops': f}
    L, q, N = case['L'], case['q'], case['N']
    nP, tab = _npairs(L), 4.0 * _npairs(L) * q * q
    if op == 'sweep':
        return {'bytes': 2.0 * N * L + tab, 'flops': 2.0 * (L - 1) * N * case['nsteps']}
    if op == 'measure':
        return {'bytes': N * (L + 4.0) + 3 * tab, 'flops': 2.0 * N * nP}
    if op == 'bicounts':
        return {'bytes': N * float(L) + 2 * tab, 'flops': 1.0 * N * nP}
    if op == 'energies':
        return {'bytes': N * (L + 4.0) + tab, 'flops': 1.0 * N * nP}
    if op in ('newton', 'iterate'):
        # an iteration reads J, dJ, bi and its target and writes dJ and bi; the sequences are needed before and after the weights
        return {'bytes': case['steps'] * (N * (2.0 * L + 8.0) + 6 * tab), 'flops': case['steps'] * 2.0 * N * nP}
    H, Lq = case['H'], L * q
    if op == 'train':
        par = Lq * H * 2 + H * H + 2 * H + Lq
        return {'bytes': 4.0 * par * 7 + N * (L + 4.0), 'flops': 6.0 * N * (H * H + H * Lq) + 4.0 * N * L * H}
    # the masks leave half of each product; the walkers and their proposals are scored and their energies taken
    return {'bytes': 4.0 * (2 * Lq * H + H * H) + tab + N * (4.0 * L + 24.0),
            'flops': 2.0 * (N * (H * H + H * Lq) + N * L * H / 2 + N * nP)}


# ---- inputs -------------------------------------------------------------------------------------------------------------

def _npairs(L):
    return L * (L - 1) // 2


def _models(case):
    return [tuple(int(x) for x in m.split('x')) for m in case['models'].split(',')]


def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1000 + salt)
    return g


def _sites(L, q, seed):
    """Site frequencies (L, q) of an alignment: a few common letters a site, none absent."""
    a = torch.rand(L, q, generator=_gen(seed, 1), device=DEV, dtype=torch.float64)
    f = (-torch.log(a.clamp_min(1e-12))) ** 2 + 0.02
    return f / f.sum(1, keepdim=True)


def _seqs(L, q, N, seed):
    """Site-major sequences (L, N) of independent sites."""
    c = torch.cumsum(_sites(L, q, seed), 1).float()
    out = torch.empty(L, N, dtype=torch.uint8, device=DEV)
    g = _gen(seed, 2)
    for i in range(L):
        out[i] = torch.searchsorted(c[i], torch.rand(N, generator=g, device=DEV)).clamp_(max=q - 1).to(torch.uint8)
    return out


def _pairs(L):
    i, j = torch.triu_indices(L, L, 1, device=DEV)
    return i, j


def _couplings(L, q, seed, sd=0.05):
    """Packed couplings: weak random pair terms plus the fields -log f, spread over the pairs."""
    h = -torch.log(_sites(L, q, seed)).float()
    h = (h - h.mean(1, keepdim=True)) / max(1, L - 1)
    i, j = _pairs(L)
    J = sd * torch.randn(len(i), q, q, generator=_gen(seed, 3), device=DEV)
    return (J + h[i][:, :, None] + h[j][:, None, :]).reshape(len(i), q * q)


def _target(L, q, seed):
    """Target bimarginals: the sites' products, with correlations."""
    f = _sites(L, q, seed).float()
    i, j = _pairs(L)
    t = f[i][:, :, None] * f[j][:, None, :]
    t = t * torch.exp(0.2 * torch.randn(t.shape, generator=_gen(seed, 4), device=DEV))
    t = t.reshape(len(i), q * q) + 1e-6
    return t / t.sum(1, keepdim=True)


class _Memory:
    """Device memory of the engine; `owner` lives as long as a tensor of it does."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {'shape': shape, 'typestr': typestr, 'data': (ptr, False), 'version': 3,
                                         'strides': None}


def _tensor(ptr, shape, typestr, owner):
    return torch.as_tensor(_Memory(ptr.value, tuple(shape), typestr, owner), device=DEV)


def _buffer(g, name, shape, typestr):
    p = ctypes.c_void_p()
    check(g._ctx, lib().mi3_buf_device_ptr(g._ctx, name.encode(), ctypes.byref(p)))
    return _tensor(p, shape, typestr, g)


def _engine(case, seed, N):
    d = tempfile.TemporaryDirectory()
    g = MCMCGPU((0, 0, None, None), case['L'], case['q'], N, WGSIZE, Path(d.name), 1024, seed)
    g._keep = d
    return g


def _put_seqs(g, name, seqs, n=None):
    """Sequences that are on the GPU already go into a buffer of the engine."""
    g.wait()
    ld = g._large_ld if name == 'seq large' else g.nseq['main']
    _buffer(g, name, (g.L, ld), '|u1')[:, :seqs.shape[1]].copy_(seqs)
    torch.cuda.synchronize()
    check(g._ctx, lib().mi3_buf_mark_written(g._ctx, name.encode()))


def _walkers(g, case, seed):
    _put_seqs(g, 'seq main', _seqs(case['L'], case['q'], case['N'], seed))


def _jstep(g, case, seed):
    """The buffers of a quasi-Newton phase."""
    L, q = case['L'], case['q']
    g.initJstep()
    target = _target(L, q, seed).cpu().numpy()
    g.setBuf('J', _couplings(L, q, seed).cpu().numpy())
    g.setBuf('bi target', target)
    _walkers(g, case, seed)
    return target


def _made(case, seed):
    """A network in mid-training: weights, and moments of the size of its gradients."""
    L, q, H = case['L'], case['q'], case['H']
    f = _sites(L, q, seed).cpu().numpy()
    return MADE(L, q, H, max_batch=case['N'], seed=seed, unimarg=f)


def _moments(case, seed):
    L, q, H = case['L'], case['q'], case['H']
    sizes = {'W1t': (L * q, H), 'b1': (H,), 'W2': (H, H), 'b2': (H,), 'W3': (L * q, H), 'b3': (L * q,)}
    g = _gen(seed, 5)
    m = {k: 1e-3 * torch.randn(s, generator=g, device=DEV) for k, s in sizes.items()}
    v = {k: 1e-6 * (0.5 + torch.rand(s, generator=g, device=DEV)) for k, s in sizes.items()}
    return m, v


STEP, RATE = 100, 1e-3    # Adam's step count and learning rate of a training step


def prepare(case, seed):
    op = case['op']
    s = SimpleNamespace(case=case, op=op)
    if op == 'batch':
        ms = _models(case)
        s.batch = PottsBatch([m[0] for m in ms], [m[1] for m in ms], [m[2] for m in ms], seed=seed)
        for k, (L, q, N) in enumerate(ms):
            s.batch.set_couplings(k, _couplings(L, q, seed + 17 * k).cpu().numpy())
            s.batch.set_seqs(k, _seqs(L, q, N, seed + 17 * k).T.contiguous().cpu().numpy())
        return s
    L, q, N = case['L'], case['q'], case['N']
    nP, qq = _npairs(L), q * q
    if op == 'train':
        s.made = _made(case, seed)
        mem = s.made.mem
        m, v = _moments(case, seed)
        M = dict(zip(('W1t', 'W2', 'W3'), made_masks(L, q, case['H'])))
        for k in PARAMS:
            mask = torch.from_numpy(M[k]).to(DEV) if k in M else 1.0
            _tensor(mem['m_' + k], m[k].shape, '<f4', mem).copy_(m[k] * mask)
            _tensor(mem['v_' + k], v[k].shape, '<f4', mem).copy_(v[k])
        s.made.t = STEP
        mem.alloc('batch', (L, N), 'u1')
        mem.sync()
        _tensor(mem['batch'], (L, N), '|u1', mem).copy_(_seqs(L, q, N, seed))
        s.out = [_tensor(mem['nll'], (N,), '<f4', mem)]
        for pre in ('', 'g_'):
            s.out += [_tensor(mem[pre + k], s.made.shape[k], '<f4', mem) for k in PARAMS]
        torch.cuda.synchronize()
        return s
    if op in ('bicounts', 'energies'):
        g = s.g = _engine(case, seed, 512)
        g.initLargeBufs(N)
        g.gen_indep('large')
        _put_seqs(g, 'seq large', _seqs(L, q, N, seed))
        if op == 'energies':
            g.setBuf('J', _couplings(L, q, seed).cpu().numpy())
            s.out = [_buffer(g, 'E large', (N,), '<f4')]
        else:
            s.out = [_buffer(g, 'bicount', (nP, qq), '<i4'), _buffer(g, 'bi', (nP, qq), '<f4')]
        return s
    g = s.g = _engine(case, seed, N)
    if op in ('newton', 'iterate'):
        s.target = _jstep(g, case, seed)
        s.node = GPU_node([g])
        s.param = SimpleNamespace(bimarg=s.target, gamma0=GAMMA, pcdamping=PC, newtonSteps=case['steps'], fracNeff=0.2,
                                  nwalkers=N, reg='l1z', regarg=(LAM,), distribute_jstep='all', beta=None)
        if op == 'newton':
            g.calcBicounts('main')
            g.bicounts_to_bimarg('main')
            s.out = [_buffer(g, 'dJ', (nP, qq), '<f4'), _buffer(g, 'E main', (N,), '<f4'),
                     _buffer(g, 'weights', (N,), '<f4'), _buffer(g, 'bi', (nP, qq), '<f4')]
        return s
    g.setBuf('J', _couplings(L, q, seed).cpu().numpy())
    _walkers(g, case, seed)
    if op == 'sweep':
        g.initMCMC(case['nsteps'], 0, 2 ** 63)
        s.out = [_buffer(g, 'seq main', (L, N), '|u1')]
    elif op == 'measure':
        s.out = [_buffer(g, 'bicount', (nP, qq), '<i4'), _buffer(g, 'bi', (nP, qq), '<f4'),
                 _buffer(g, 'E main', (N,), '<f4')]
    else:
        s.made = _made(case, seed)
        s.mixed = MixedSampler(g, s.made, seed=seed + 1)
        s.out = [_buffer(g, n, (L, N), '|u1') for n in ('seq main', 'seq prop')] + \
                [_buffer(g, n, (N,), '<f4') for n in ('E main', 'E prop', 'made nll cur', 'made nll prop')]
    return s


def run(s):
    op = s.op
    if op == 'sweep':
        s.g.runMCMC()
        return s.out
    if op == 'batch':
        s.batch.run(s.case['nsweeps'])
        return [s.batch.get_seqs(m) for m in range(len(s.batch))]
    if op == 'measure':
        s.g.calcBicounts('main')
        s.g.bicounts_to_bimarg('main')
        s.g.calcEnergies('main')
        return s.out
    if op == 'bicounts':
        s.g.calcBicounts('large')
        s.g.bicounts_to_bimarg('large')
        return s.out
    if op == 'energies':
        s.g.calcEnergies('large')
        return s.out
    if op == 'iterate':
        n, J, bi = iterNewton(s.param, None, s.node, lambda *a: None)
        return [n, J, bi]
    if op == 'newton':
        # the driver's loop: dJ from zero, the host reads the minimum and the weights' sums of every iteration
        g, ref = s.g, 0.0
        g.fillBuf('dJ', 0)
        for _ in range(s.case['steps']):
            g.updateJ(GAMMA, PC)
            g.reg_l1z(GAMMA, PC, LAM)
            g.calcEnergies('main', 'dJ')
            g.min_buf('E main')
            low = g.getBuf('minout')
            g.dE_to_weights('main', ref)
            g.weight_statistics('main')
            sums = g.getBuf('weightstats')
            g.weightedMarg('main')
            g.renormalize_bimarg()
            stats = sums.read()
            ref = float(low.read()[0])
        return s.out + [stats]
    if op == 'train':
        s.made.loss_and_grads(s.made.mem['batch'], s.case['N'], s.case['N'])
        s.made.adam(RATE)
        return s.out
    s.mixed.propose()
    return s.out


# ---- the same in 64 bits ------------------------------------------------------------------------------------------------

def _chunks(seqs, q, most=2 ** 28):
    """One-hot rows (n, L*q) of the sequences, some at a time."""
    L, N = seqs.shape
    step = max(256, int(most / (L * q)) // 4)
    rows = torch.arange(L, device=DEV)[None, :] * q
    for n in range(0, N, step):
        s = seqs[:, n:n + step].T.long() + rows
        X = torch.zeros(s.shape[0], L * q, dtype=torch.float64, device=DEV)
        yield n, X.scatter_(1, s, 1.0)


def _square(J, L, q):
    """Packed couplings as the upper blocks of an (L*q, L*q) matrix."""
    i, j = _pairs(L)
    A = torch.zeros(L, L, q, q, dtype=torch.float64, device=DEV)
    A[i, j] = J.double().reshape(-1, q, q)
    return A.permute(0, 2, 1, 3).reshape(L * q, L * q)


def _packed(A, L, q):
    i, j = _pairs(L)
    return A.reshape(L, q, L, q).permute(0, 2, 1, 3)[i, j].reshape(-1, q * q)


def _exact_energies(seqs, J, q):
    A = _square(J, seqs.shape[0], q)
    E = torch.empty(seqs.shape[1], dtype=torch.float64, device=DEV)
    for n, X in _chunks(seqs, q):
        E[n:n + len(X)] = ((X @ A) * X).sum(1)
    return E


def _exact_marginals(seqs, w, q):
    L = seqs.shape[0]
    A = torch.zeros(L * q, L * q, dtype=torch.float64, device=DEV)
    for n, X in _chunks(seqs, q):
        A += X.T @ (X if w is None else X * w[n:n + len(X), None])
    return _packed(A, L, q)


def _exact_step(J, dJ, bi, target, q, gamma, pc, lam):
    """Coupling update and l1z step of one iteration."""
    dJ = dJ - gamma * (target - bi) / (bi + pc)
    t = (J + dJ).reshape(-1, q, q)
    J0 = (t - t.mean(2, keepdim=True) - t.mean(1, keepdim=True) + t.mean((1, 2), keepdim=True)).reshape(-1, q * q)
    R = -lam * torch.sign(J0) * gamma / (bi + pc)
    return torch.where(torch.sign(J0) != torch.sign(J0 + R), dJ - J0, dJ + R)


def exact(case, seed):
    op = case['op']
    if op in ('sweep', 'batch'):
        return None   # whole numbers only
    L, q, N = case['L'], case['q'], case['N']
    seqs = _seqs(L, q, N, seed)
    if op == 'measure':
        c = _exact_marginals(seqs, None, q)
        return [c.round().to(torch.int32), c / N, _exact_energies(seqs, _couplings(L, q, seed), q)]
    if op == 'bicounts':
        c = _exact_marginals(seqs, None, q)
        return [c.round().to(torch.int32), c / N]
    if op == 'energies':
        return [_exact_energies(seqs, _couplings(L, q, seed), q)]
    if op in ('newton', 'iterate'):
        J, target = _couplings(L, q, seed).double(), _target(L, q, seed).double()
        bi, dJ, ref = _exact_marginals(seqs, None, q) / N, torch.zeros_like(J), 0.0
        # the engine takes these as 32-bit numbers
        gamma, pc, lam = (float(np.float32(x)) for x in (GAMMA, PC, LAM))
        for _ in range(case['steps']):
            dJ = _exact_step(J, dJ, bi, target, q, gamma, pc, lam)
            E = _exact_energies(seqs, dJ, q)
            w = torch.exp(ref - E)
            F = _exact_marginals(seqs, w, q)
            bi = F / F.sum(1, keepdim=True)
            ref = float(torch.clamp(E.min(), max=0.0))
        if op == 'iterate':
            return [None, J + dJ, bi]
        return [dJ, E, w, bi, torch.stack([w.sum(), (w * w).sum()])]
    return _exact_made(case, seed, seqs)


def _exact_made(case, seed, seqs):
    L, q, H, N = case['L'], case['q'], case['H'], case['N']
    made = _made(dict(case, N=8), seed)
    P = {k: torch.from_numpy(made.get(k)).to(DEV).double() for k in PARAMS}
    made.close()
    if case['op'] == 'train':
        for k in PARAMS:
            P[k].requires_grad_(True)
    idx = seqs.T.long() + torch.arange(L, device=DEV)[None, :] * q
    nlls = []
    step = N if case['op'] == 'train' else 4096
    for n in range(0, N, step):
        X = torch.zeros(min(step, N - n), L * q, dtype=torch.float64, device=DEV).scatter_(1, idx[n:n + step], 1.0)
        h1 = torch.relu(X @ P['W1t'] + P['b1'])
        h2 = torch.relu(h1 @ P['W2'].T + P['b2'])
        z = (h2 @ P['W3'].T + P['b3']).reshape(-1, L, q)
        nlls.append((torch.logsumexp(z, 2) - (z.reshape(-1, L * q) * X).reshape(-1, L, q).sum(2)).sum(1))
    nll = torch.cat(nlls)
    if case['op'] == 'propose':
        E = _exact_energies(seqs, _couplings(L, q, seed), q)
        return [None, None, E, None, nll, None]
    nll.mean().backward()
    m, v = _moments(case, seed)
    M = dict(zip(('W1t', 'W2', 'W3'), made_masks(L, q, H)))
    new, grads = [], []
    b1, b2, eps, t = 0.9, 0.999, 1e-8, STEP + 1
    for k in PARAMS:
        mask = torch.from_numpy(M[k]).to(DEV).double() if k in M else torch.ones_like(P[k])
        raw = P[k].grad
        g = raw * mask
        mk = b1 * m[k].double() * mask + (1 - b1) * g
        vk = b2 * v[k].double() + (1 - b2) * g * g
        new.append(((P[k] - RATE * (mk / (1 - b1 ** t)) / (torch.sqrt(vk / (1 - b2 ** t)) + eps)) * mask).detach())
        grads.append(raw)
    # gradients of masked entries are whatever the dense products give: the engine's are compared as they are
    return [nll.detach()] + new + grads
