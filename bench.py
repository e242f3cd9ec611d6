#!/usr/bin/env python3
"""Benchmark of the plain Mi3 sweep on one MI355X.

Workload: the production-size inference round's sampler -- a random Potts
model with L=232 sites and q=21 letters (fields h ~ N(0,1), couplings
J ~ N(0, 0.05) moved to the zero-sum gauge and folded into the fieldless
float32 form), 2^18 walkers.  One step = one MCMC kernel call of
8 sweeps (8*L single-site Metropolis updates per walker).  The value is
site-updates/s over the timed steps, with walker state and couplings resident
in HBM before timing starts.

Printed as one JSON line, with
  energy_ess:   energy effective samples per second of the same sampler
                (walker-averaged integrated autocorrelation time of the
                per-sweep energy traces, Sokal window c=5) on an equilibrated
                ensemble;
  round:        wall seconds per inference round (MCMC of 128 sweeps,
                bicounts, the quasi-Newton phase and the per-round host work)
                of `Mi3.py infer` on target bimarginals sampled from the same
                model, with and without the bz2 sequence write;
  roofline:     algorithmic bytes (L+1 per site update: read the walker's L
                residues, write back one) per launch over the launch duration
                measured with HIP events on the engine's stream, against the
                8 TB/s HBM peak, and against the best bandwidth plain
                streaming (copies, a read-only stream) reaches in the same run
                (achievable);
  cpu_baseline: the CPU port of the same sampler (oracle/oracle.c, float32
                as the reference CPU sampler) on this host's cores, on a
                bounded sample of the same workload.
"""
import argparse
import json
import os
import sys
import tempfile
import time
from pathlib import Path

import numpy as np

REPO = Path(__file__).resolve().parent
sys.path.insert(0, str(REPO / 'mi3-gpu_amd'))
sys.path.insert(0, str(REPO))

METRIC = "site-updates/s & energy-ESS/s at L=232 q=21; s per inference round at fixed SSR"
HBM_PEAK_GBS = 8000.0

# HBM bytes per k_sweep launch, measured with two rocprofv3 --pmc runs
# (FETCH_SIZE, then WRITE_SIZE, KiB per dispatch) of
# `bench.py --steps 2 --warmup 1 --no-cpu --ess-sweeps 0 --rounds 0
# --copy-calibration 1024`, each counter scaled by what it reads for a 1 GiB
# device-to-device copy in the same run (FETCH_SIZE x2.0, WRITE_SIZE x1.0);
# summary in profiles/k_sweep_L232_q21_N262144_pmc_traffic.md.  Keyed by
# (L, q, walkers, sweeps per launch, walkers per work-group).
MEASURED_TRAFFIC = {(232, 21, 2 ** 18, 8, 512): 13.41e9}

# VALU issue of the same k_sweep launch from SQ counters
# (SQ_ACTIVE_INST_VALU per CU over SQ_BUSY_CYCLES; summary and command in
# profiles/k_sweep_L232_q21_N262144_kernel_trace.md).  Same key.
MEASURED_VALU_BUSY = {(232, 21, 2 ** 18, 8, 512): 0.69}


def host_cores():
    """Cores this job may use: its CPU affinity, capped by OMP_NUM_THREADS
    when the host sets it (the share a shared GPU host gives one job)."""
    n = len(os.sched_getaffinity(0)) if hasattr(os, 'sched_getaffinity') else os.cpu_count()
    omp = os.environ.get('OMP_NUM_THREADS')
    if omp and omp.isdigit() and int(omp) > 0:
        n = min(n, int(omp))
    return max(1, int(n or 1))


def production_model(L=232, q=21, seed=1, hs=1.0, js=0.05):
    """h ~ N(0,hs), J ~ N(0,js), zero-sum gauge, folded to fieldless float32."""
    from mi3gpu.utils.changeGauge import zeroJGauge, fieldlessGaugeEven
    rng = np.random.default_rng(seed)
    h = rng.normal(0, hs, size=(L, q))
    J = rng.normal(0, js, size=(L * (L - 1) // 2, q * q))
    h, J = zeroJGauge(h, J)
    return fieldlessGaugeEven(h, J)[1].astype('<f4')


def _pf_class(q):
    """float4 loads per thread per staged coupling chunk (launch.h pf_class)."""
    need = (q * q * 32 // 4 + 511) // 512
    return 1 if need <= 1 else 4 if need <= 4 else 7 if need <= 7 else 10


def cpu_baseline(J, L, q, seed, target_s=20.0):
    """Time the CPU port of the sampler on this host's cores."""
    from oracle import cboracle
    nthr = host_cores()
    walkers = 64 * nthr
    rng = np.random.default_rng(seed)
    s = rng.integers(0, q, size=(walkers, L)).astype('<u1')
    t0 = time.perf_counter()
    s = cboracle.metropolis_f32(s, J, seed, 0, L, nthreads=nthr)
    t1 = time.perf_counter() - t0
    sweeps = int(max(1, min(4096, target_s / max(t1, 1e-3))))
    t0 = time.perf_counter()
    cboracle.metropolis_f32(s, J, seed, 2 * L, sweeps * L, nthreads=nthr)
    dt = time.perf_counter() - t0
    su = walkers * sweeps * L
    return {"value": su / dt, "unit": "site-updates/s", "cores": nthr, "kind": "port",
            "sample": f"{walkers} walkers x {sweeps} sweeps of the same L=232 q=21 model "
                      f"({su:.3g} site updates, {dt:.1f} s, oracle/oracle.c float32, "
                      f"{nthr} OpenMP threads)"}


ALPHA21 = '-ACDEFGHIKLMNPQRSTVWY'


def sample_target(J, L, q, n, sweeps, seed, wgsize):
    """Sample n sequences of the model (sweeps sweeps from uniform random
    sequences); returns (seqs (n, L) u8, bimarg with Jeffreys pseudocount)."""
    from mi3gpu.mcmcGPU import MCMCGPU
    from mi3gpu.utils.pseudocount import mutation_pc
    with tempfile.TemporaryDirectory() as d:
        g = MCMCGPU((0, 0, None, None), L, q, n, wgsize, Path(d), 1024, seed)
        g.initMCMC(8 * L, 0, 2 ** 63)
        g.setBuf('J', J)
        g.setBuf('seq main', np.random.default_rng(seed).integers(0, q, size=(n, L)).astype('u1'))
        for _ in range(max(1, sweeps // 8)):
            g.runMCMC()
        g.calcBicounts('main')
        bc = g.getBuf('bicount').read()
        seqs = g.getBuf('seq main').read()
        del g
    f = bc.astype(np.float64) / n
    return seqs, mutation_pc(f, n).astype('<f4')


def measure_ess(J, seqs, L, q, T, seed, wgsize):
    """Energy traces of T single-sweep launches from an equilibrated
    ensemble; returns the energy-ESS figures."""
    from mi3gpu.mcmcGPU import MCMCGPU
    from mi3gpu.utils.ess import energy_ess
    n = seqs.shape[0]
    with tempfile.TemporaryDirectory() as d:
        g = MCMCGPU((0, 0, None, None), L, q, n, wgsize, Path(d), 1024, seed, profile=True)
        g.initMCMC(L, 0, 2 ** 63)
        g.setBuf('J', J)
        g.setBuf('seq main', seqs)
        g.profile_reset()
        E = np.empty((T, n), dtype=np.float32)
        for t in range(T):
            g.runMCMC()
            g.calcEnergies('main')
            E[t] = g.getBuf('E main').read()
        kms, kcnt = g.kernel_ms('mcmc')
        del g
    ess, tau, W = energy_ess(E)
    t_sample = kms * kcnt * 1e-3
    half = T // 2
    return {"value": ess / t_sample, "unit": "energy effective samples/s",
            "tau_int_sweeps": tau, "window": W, "walkers": n, "sweeps": T,
            "ess": ess, "sampling_s": t_sample,
            "mean_E_first_half": float(E[:half].mean()),
            "mean_E_second_half": float(E[half:].mean())}


def _print_round(r):
    print(f"{r['run']}: {r['wall_s']:.2f} s, SSR {r['ssr']:.4f}, "
          f"{r['newton_steps']} Newton steps, {r['equil_launches']} equilibration launches",
          file=sys.stderr, flush=True)


def measure_rounds(target, L, q, N, rounds, seed, equiltime='8', nsteps=None):
    """`Mi3.py infer` rounds at the production size; per-round wall times.
    Default schedule: 8 launches of 16 sweeps (128 sweeps per round);
    equiltime 'auto' uses the reference's equilibration test instead."""
    import mi3gpu.Mi3 as Mi3
    with tempfile.TemporaryDirectory() as d:
        np.save(Path(d) / 'target.npy', target)
        args = ['infer', '--init_model', 'independent', '--bimarg', str(Path(d) / 'target.npy'),
                '--alpha=' + ALPHA21[:q], '--nwalkers', str(N),
                '--nsteps', str(nsteps or 16 * L), '--equiltime', str(equiltime),
                '--mcsteps', str(rounds), '--rngseed', str(seed),
                '--outdir', str(Path(d) / 'infer')]
        import contextlib
        import mi3gpu.NewtonSteps as NS
        NS.round_hook = _print_round
        # Mi3's own log lines go to stderr; stdout keeps the one JSON line
        try:
            with contextlib.redirect_stdout(sys.stderr):
                p = Mi3.main(args)
        finally:
            NS.round_hook = None
        st = p.round_stats
    floor = float(np.sum(target * (1 - target)) / N)
    wall = [r['wall_s'] for r in st]
    nowrite = [r['wall_s'] - r['status_write_s'] for r in st]
    # the first round whose SSR is within twice the sampling floor
    at = next((k for k, r in enumerate(st) if r['ssr'] <= 2 * floor), None)
    return {"value": float(np.mean(wall)), "unit": "s/round",
            "s_per_round_without_seq_write": float(np.mean(nowrite)),
            "rounds": st, "ssr_floor": floor,
            "fixed_ssr": None if at is None else {
                "round": at, "ssr": st[at]['ssr'], "s": st[at]['wall_s'],
                "s_without_seq_write": st[at]['wall_s'] - st[at]['status_write_s'],
                "cumulative_s": float(np.sum(wall[:at + 1]))},
            "note": "rounds from the independent-site model; SSR per round; fixed_ssr is the "
                    "first round with SSR <= 2 x floor (null if not reached)"}


# The reference's published end-to-end result (UserGuide.md:103-113): the
# HIV protease run of examples/HIV_inference/pbs.sh:11-20, rounds run_04..06
# and run_63 (Ferr is the mean relative error over target bimarginals
# above 0.01, the log's rel% / 100).
HIV_PUBLISHED = {4: {'jstep': 4092, 'ssr': 0.206, 'ferr': 0.00992, 'X': -119.709, 'Xo': -122.201},
                 5: {'jstep': 5115, 'ssr': 0.204, 'ferr': 0.00984, 'X': -120.186, 'Xo': -122.374},
                 6: {'jstep': 6138, 'ssr': 0.203, 'ferr': 0.00971, 'X': -120.275, 'Xo': -122.534},
                 63: {'ssr': 0.010, 'ferr': 0.00856, 'X': -10.118, 'Xo': -10.878}}


def measure_hiv(rounds, walkers=2 ** 18, seed=7):
    """`Mi3.py infer` with the settings of the reference's HIV example
    (examples/HIV_inference/pbs.sh:11-20: independent start, 2^18 walkers,
    damping 0.01, l1z 1e-4, 64 rounds; reference defaults otherwise --
    nsteps 2048, equiltime auto, newtonsteps 1024, gamma 4e-4) on the
    reference's target (L=93, q=4).  Per-round SSR, Ferr, X and wall time
    beside the published values, and the first round within twice the SSR
    floor sum f(1-f)/N."""
    import contextlib
    import mi3gpu.Mi3 as Mi3
    target = np.load(REPO / 'tests' / 'golden' / 'hiv_bimarg_pc.npy')
    with tempfile.TemporaryDirectory() as d:
        args = ['infer', '--init_model', 'independent',
                '--bimarg', str(REPO / 'tests' / 'golden' / 'hiv_bimarg_pc.npy'),
                '--alpha', 'ABCD', '--nwalkers', str(walkers), '--damping', '0.01',
                '--mcsteps', str(rounds), '--reg', 'l1z:0.0001', '--rngseed', str(seed),
                '--outdir', str(Path(d) / 'hiv')]
        t0 = time.perf_counter()
        import mi3gpu.NewtonSteps as NS
        NS.round_hook = _print_round
        try:
            with contextlib.redirect_stdout(sys.stderr):
                p = Mi3.main(args)
        finally:
            NS.round_hook = None
        total = time.perf_counter() - t0
    st = p.round_stats
    floor = float(np.sum(target * (1 - target)) / walkers)
    at = next((k for k, r in enumerate(st) if r['ssr'] <= 2 * floor), None)
    keep = ('ssr', 'ferr', 'X', 'Xo', 'jstep', 'newton_steps', 'equil_launches', 'wall_s',
            'mcmc_s', 'newton_s', 'status_write_s')
    per_round = [{k: r[k] for k in keep} for r in st]
    compare = {f"run_{k:02d}": {"published": v, "measured": per_round[k]}
               for k, v in HIV_PUBLISHED.items() if k < len(per_round)}
    wall = [r['wall_s'] for r in st]
    return {"workload": "Mi3.py infer, examples/HIV_inference/pbs.sh settings, L=93 q=4, "
                        f"{walkers} walkers, {rounds} rounds, reference defaults",
            "rounds": per_round, "published_vs_measured": compare, "ssr_floor": floor,
            "s_per_round": float(np.mean(wall)),
            "s_per_round_without_seq_write": float(np.mean(
                [r['wall_s'] - r['status_write_s'] for r in st])),
            "total_s": total,
            "fixed_ssr": None if at is None else {
                "round": at, "ssr": st[at]['ssr'], "s": st[at]['wall_s'],
                "s_without_seq_write": st[at]['wall_s'] - st[at]['status_write_s'],
                "cumulative_s": float(np.sum(wall[:at + 1]))}}


def measure_batch(rounds, sweeps=64, nmodels=64, seed=4):
    """Batched uneven models: nmodels Potts models with L ~ U{50..400},
    q in {4, 21} (probability 1/2 each), h ~ N(0,1), J ~ N(0,0.05) in the
    zero-sum gauge folded to fieldless float32, 512*L walkers each, `sweeps`
    sweeps per round in one graph launch, tiles chosen by the autotuner."""
    from mi3gpu.batch import PottsBatch
    rng = np.random.default_rng(seed)
    Ls = rng.integers(50, 401, size=nmodels)
    qs = np.where(rng.random(nmodels) < 0.5, 4, 21)
    Ns = 512 * Ls
    b = PottsBatch(Ls, qs, Ns, seed=seed)
    for m, (L, q) in enumerate(zip(Ls, qs)):
        b.set_couplings(m, production_model(int(L), int(q), seed=1000 + m))
        b.set_seqs(m, rng.integers(0, q, size=(int(512 * L), int(L))).astype('u1'))
        if m % 16 == 15:
            print(f"batch: {m + 1} models set up", file=sys.stderr, flush=True)
    t0 = time.perf_counter()
    b.tune(1)
    b.wait()
    t_tune = time.perf_counter() - t0
    print(f"batch: tuned in {time.perf_counter() - t0:.1f} s", file=sys.stderr, flush=True)
    b.run(sweeps)                 # capture + one warm round
    b.wait()
    print("batch: warm round done", file=sys.stderr, flush=True)
    t0 = time.perf_counter()
    for _ in range(rounds):
        b.run(sweeps)
    b.wait()
    dt = (time.perf_counter() - t0) / rounds
    su = float(sum(int(n) * int(L) * sweeps for n, L in zip(Ns, Ls)))
    tiles = {}
    for m, (L, q) in enumerate(zip(Ls, qs)):
        key = f"L{'<=128' if L <= 128 else ('<=256' if L <= 256 else '>256')} q={q}"
        tiles[key] = b.tile(m)
    b.close()
    return {"value": su / dt, "unit": "site-updates/s", "s_per_round": dt, "rounds": rounds,
            "models": nmodels, "sweeps_per_round": sweeps, "walkers": int(Ns.sum()),
            "site_updates_per_round": su, "tiles": tiles, "tune_s": t_tune,
            "workload": "64 models, L~U{50..400}, q in {4,21}, 512*L walkers each, "
                        "64 sweeps per round in one HIP graph"}


def measure_kernels(n=2 ** 20, L=232, q=21, reps=3):
    """Bimarginal counts (4-bit one-hot Gram product on the matrix cores) and
    batch energies standalone on n uniform i.i.d. sequences: average kernel
    time (HIP events) and rates.  Useful MACs of the counts:
    n*q^2*L(L-1)/2; energies: n*L(L-1)/2 coupling gathers."""
    from mi3gpu.mcmcGPU import MCMCGPU
    J = production_model(L, q, seed=1)
    seqs = np.random.default_rng(3).integers(0, q, size=(n, L)).astype('u1')
    with tempfile.TemporaryDirectory() as d:
        g = MCMCGPU((0, 0, None, None), L, q, n, 512, Path(d), 1024, 2, profile=True)
        g.setBuf('J', J)
        g.setBuf('seq main', seqs)
        g.calcBicounts('main')
        g.calcEnergies('main')
        g.wait()
        g.profile_reset()
        for r in range(reps):
            g.calcBicounts('main')
            g.calcEnergies('main')
            g.wait()
            print(f"kernels: bicounts + energies, repetition {r + 1} of {reps}",
                  file=sys.stderr, flush=True)
        bc_ms, _ = g.kernel_ms('calcBicounts')
        en_ms, _ = g.kernel_ms('getEnergies')
        bc = g.getBuf('bicount').read()
        del g
    nP = L * (L - 1) // 2
    macs = float(n) * q * q * nP
    ok_rows = bool(np.all(bc.sum(axis=1) == n))
    return {"sequences": n, "L": L, "q": q,
            "bicounts_ms": bc_ms, "bicounts_TOPS": 2 * macs / (bc_ms * 1e-3) / 1e12,
            "bicounts_frac_of_10_POPS": 2 * macs / (bc_ms * 1e-3) / 10.0e15,
            "bicount_rows_sum_to_n": ok_rows,
            "energies_ms": en_ms, "energy_gathers_per_s": float(n) * nP / (en_ms * 1e-3)}


def measure_newton_kernels(n=2 ** 18, L=232, q=21, reps=5, seed=9):
    """One quasi-Newton iteration's kernels at the production walker count
    on equal-weight-ish Zwanzig weights: energies under a dJ, weights, and
    weighted marginals, average kernel time (HIP events).  Rates: energies
    in coupling gathers (n*L(L-1)/2 per call) and L2->LDS staging bytes;
    weighted marginals in 64-bit LDS bin additions (n*L(L-1)/2 per call)."""
    from mi3gpu.mcmcGPU import MCMCGPU
    rng = np.random.default_rng(seed)
    nP = L * (L - 1) // 2
    J = production_model(L, q, seed=1)
    dJ = rng.normal(0, 1e-3, size=(nP, q * q)).astype('<f4')
    seqs = rng.integers(0, q, size=(n, L)).astype('u1')
    with tempfile.TemporaryDirectory() as d:
        g = MCMCGPU((0, 0, None, None), L, q, n, 512, Path(d), 1024, 2, profile=True)
        g.initJstep()
        g.setBuf('J', J)
        g.setBuf('dJ', dJ)
        g.setBuf('seq main', seqs)

        def iteration():
            g.calcEnergies('main', 'dJ')
            g.min_buf('E main')
            g.dE_to_weights('main', 0.0)
            g.weight_statistics('main')
            g.weightedMarg('main')

        iteration()
        g.wait()
        g.profile_reset()
        for r in range(reps):
            iteration()
            g.wait()
            print(f"kernels: quasi-Newton iteration {r + 1} of {reps}", file=sys.stderr,
                  flush=True)
        en_ms, _ = g.kernel_ms('getEnergies')
        wm_ms, _ = g.kernel_ms('weightedMarg')
        # the weighted marginals' 64-bit LDS atomic adds alone (same
        # work-group size, histogram and column pattern, no loads)
        from mi3gpu._lib import lib, check
        ap_wgs, ap_iters = 8 * 256, 2048
        for _ in range(4):
            check(g._ctx, lib().mi3_wm_atomic_probe(g._ctx, ap_wgs, ap_iters))
        g.wait()
        g.profile_reset()
        for _ in range(3):
            check(g._ctx, lib().mi3_wm_atomic_probe(g._ctx, ap_wgs, ap_iters))
        g.wait()
        ap_ms, _ = g.kernel_ms('wmAtomicProbe')
        ceiling = ap_wgs * 1024.0 * ap_iters / (ap_ms * 1e-3)
        del g
    units = sum(max(0, (L + 31) // 32 - (i + 1) // 32) for i in range(L - 1))
    chunk_bytes = _pf_class(q) * 512 * 16
    stage = (n // 512) * units * chunk_bytes
    return {"sequences": n, "L": L, "q": q,
            "energies_ms": en_ms, "energy_gathers_per_s": float(n) * nP / (en_ms * 1e-3),
            "energies_staging_bytes": stage,
            "energies_staging_TBps": stage / (en_ms * 1e-3) / 1e12,
            "weighted_marg_ms": wm_ms,
            "weighted_marg_u64_adds_per_s": float(n) * nP / (wm_ms * 1e-3),
            "weighted_marg_atomic_ceiling_adds_per_s": ceiling,
            "weighted_marg_frac_of_atomic_ceiling": float(n) * nP / (wm_ms * 1e-3) / ceiling}


def _best_wgsize(J, s0, L, q, seed):
    """Walkers per work-group with the fastest single sweep for this walker
    count (128 / 256 / 512), from three timed launches each."""
    from mi3gpu.mcmcGPU import MCMCGPU
    best = None
    for wg in (128, 256, 512):
        with tempfile.TemporaryDirectory() as d:
            g = MCMCGPU((0, 0, None, None), L, q, len(s0), wg, Path(d), 1024, seed)
            g.initMCMC(L, 0, 2 ** 63)
            g.setBuf('J', J)
            g.setBuf('seq main', s0)
            g.runMCMC()
            g.wait()
            t0 = time.perf_counter()
            for _ in range(3):
                g.runMCMC()
            g.wait()
            dt = time.perf_counter() - t0
            del g
        if best is None or dt < best[1]:
            best = (wg, dt)
    return best[0]


def measure_made(J, seqs, L, q, ntrain=2 ** 18, N=2 ** 16, H=512, train_steps=1500,
                 batch=4096, lr=1e-3, ratio=8, plain_sweeps=128, cycles=48, timed=8, seed=7):
    """Learned proposal against the plain sweep on the same GPU and walkers.

    A MADE (L*q -> H -> H -> L*q, bf16 matrix-core products) is trained by
    Adam on `ntrain` equilibrated MCMC sequences of the model; N walkers
    (other equilibrated sequences) then run cycles of `ratio` sweeps followed
    by one independence Metropolis-Hastings step with MADE proposals.  Both
    forms are timed by wall clock over whole cycles (sweeps, energies,
    proposals), and their energy traces (per sweep for the plain form, per
    cycle for the mixed one) give the integrated autocorrelation time;
    energy-ESS/s = N / (2 tau t_interval)."""
    from mi3gpu.mcmcGPU import MCMCGPU
    from mi3gpu.made import MADE, MixedSampler
    from mi3gpu.utils.ess import energy_ess
    train, s0 = seqs[:ntrain], seqs[ntrain:ntrain + N]
    wg = _best_wgsize(J, s0, L, q, seed)
    f1 = np.stack([np.bincount(train[:, i], minlength=q) for i in range(L)]) / len(train)
    made = MADE(L, q, H, max_batch=N, seed=seed, unimarg=f1)
    made.mem.alloc('train', (L, ntrain), 'u1')
    made.mem.write('train', np.ascontiguousarray(train.T))
    made.mem.alloc('heldout', (L, N), 'u1')
    made.mem.write('heldout', np.ascontiguousarray(s0.T))
    made.mem.alloc('heldout nll', (N,), 'f4')
    made.mem.sync()
    t0 = time.perf_counter()
    hist = made.train(made.mem['train'], ntrain, ntrain, steps=train_steps, batch=batch, lr=lr,
                      seed=seed, log_every=max(1, train_steps // 6))
    t_train = time.perf_counter() - t0
    print(f"MADE trained: {train_steps} steps in {t_train:.1f} s, nll {hist[-1][1]:.3f}",
          file=sys.stderr, flush=True)
    made.nll(made.mem['heldout'], N, N, made.mem['heldout nll'])
    heldout = float(np.mean(made.get('heldout nll')))

    def run(mixed, T):
        with tempfile.TemporaryDirectory() as d:
            g = MCMCGPU((0, 0, None, None), L, q, N, wg, Path(d), 1024, seed + 1)
            g.initMCMC(L, 0, 2 ** 63)
            g.setBuf('J', J)
            g.setBuf('seq main', s0)
            ms = MixedSampler(g, made, seed=seed + 2) if mixed else None

            def interval():
                if mixed:
                    for _ in range(ratio):
                        g.runMCMC()
                    ms.propose()
                else:
                    g.runMCMC()
                    g.calcEnergies('main')

            interval()
            g.wait()
            n_timed = timed if mixed else timed * ratio
            t0 = time.perf_counter()
            for _ in range(n_timed):
                interval()
            g.wait()
            t_int = (time.perf_counter() - t0) / n_timed
            E = np.empty((T, N), np.float32)
            for t in range(T):
                interval()
                E[t] = g.getBuf('E main').read()
            acc = ms.accepted() / (N * (T + n_timed + 1)) if mixed else None
            if mixed:   # cost of the proposal step alone
                g.wait()
                t0 = time.perf_counter()
                for _ in range(3):
                    ms.propose()
                g.wait()
                t_prop = (time.perf_counter() - t0) / 3
            del g
        ess, tau, W = energy_ess(E)
        r = {"energy_ess_per_s": N / (2 * tau * t_int), "tau_int": tau, "window": W,
             "interval_ms": t_int * 1e3, "traced_intervals": T,
             "mean_E": float(E.mean()), "sem_E": float(E.mean(axis=0).std() / np.sqrt(N) *
                                                       np.sqrt(2 * tau))}
        if mixed:
            r.update(acceptance=acc, proposal_step_ms=t_prop * 1e3)
        return r

    plain = run(False, plain_sweeps)
    print(f"plain: tau {plain['tau_int']:.2f} sweeps", file=sys.stderr, flush=True)
    mixed = run(True, cycles)
    print(f"mixed: tau {mixed['tau_int']:.2f} cycles, acceptance {mixed['acceptance']:.3f}",
          file=sys.stderr, flush=True)
    made.close()
    # the mixed form's ceiling at this proposal cost: with every proposal
    # accepted the energy decorrelates each cycle (tau = 1/2 cycle), so
    # energy-ESS/s = N / t_cycle against the plain N / (2 tau t_sweep)
    t_sweep, t_prop = plain["interval_ms"], mixed["proposal_step_ms"]
    bound = 2 * plain["tau_int"] * t_sweep / (ratio * t_sweep + t_prop)
    return {"value": mixed["energy_ess_per_s"], "unit": "energy effective samples/s",
            "vs_plain": mixed["energy_ess_per_s"] / plain["energy_ess_per_s"],
            "vs_plain_bound_all_accepted": bound,
            "plain": dict(plain, interval="1 sweep"),
            "mixed": dict(mixed, interval=f"{ratio} sweeps + 1 MADE proposal per walker"),
            "walkers": N, "walkers_per_workgroup": wg,
            "made": {"H": H, "train_sequences": ntrain, "train_steps": train_steps,
                     "batch": batch, "lr": lr, "train_s": t_train,
                     "nll_history": hist, "heldout_nll": heldout}}


def measure_config1(seed=0):
    """The reference's CPU-runnable round: L=99, q=4, h ~ N(0,0.5),
    J ~ N(0,0.1) (zero-sum gauge, fieldless float32); target bimarginals of
    10,000 sequences after 2^14 sweeps (+ Jeffreys pseudocount); one round of
    16,384 walkers x 64 sweeps + bicounts + quasi-Newton phase (reference
    defaults).  GPU: `Mi3.py infer`, one round, wall time.  CPU: the
    reference path's parts timed on this host -- the sampler (C port,
    OpenMP), numpy bicounts (one core) and numpy quasi-Newton iterations (one
    core; two timed, scaled by the GPU round's iteration count)."""
    import contextlib
    import io
    import mi3gpu.Mi3 as Mi3
    from mi3gpu.mcmcGPU import MCMCGPU
    from mi3gpu.utils.pseudocount import mutation_pc
    from oracle import cboracle, potts_oracle as po
    L, q, N = 99, 4, 16384
    J = production_model(L, q, seed=seed, hs=0.5, js=0.1)
    with tempfile.TemporaryDirectory() as d:
        nt = 10240
        g = MCMCGPU((0, 0, None, None), L, q, nt, 512, Path(d), 1024, seed)
        g.initMCMC(64 * L, 0, 2 ** 63)
        g.setBuf('J', J)
        g.setBuf('seq main', np.random.default_rng(seed).integers(0, q, (nt, L)).astype('u1'))
        for _ in range(2 ** 14 // 64):
            g.runMCMC()
        tseq = g.getBuf('seq main').read()[:10000]
        del g
        f = cboracle.bicounts(tseq, q).astype(np.float64) / 10000
        target = mutation_pc(f, 10000).astype('<f4')
        np.save(Path(d) / 'target.npy', target)
        args = ['infer', '--init_model', 'independent', '--bimarg', str(Path(d) / 'target.npy'),
                '--alpha', 'ABCD', '--nwalkers', str(N), '--nsteps', str(8 * L),
                '--equiltime', '8', '--mcsteps', '1', '--rngseed', '7',
                '--outdir', str(Path(d) / 'infer')]
        with contextlib.redirect_stdout(io.StringIO()):
            p = Mi3.main(args)
        gpu = p.round_stats[0]
        # CPU parts on the same sizes
        nthr = host_cores()
        s0 = np.random.default_rng(1).integers(0, q, (N, L)).astype('u1')
        t0 = time.perf_counter()
        s1 = cboracle.metropolis_f32(s0, J, 7, 0, 64 * L, nthreads=nthr)
        t_samp = time.perf_counter() - t0
        t0 = time.perf_counter()
        bc = po.bicounts(s1, q)
        t_bc = time.perf_counter() - t0
        t0 = time.perf_counter()
        it, *_ = po.iter_newton(s1, J, target, 4e-4, 1e-3, 4, 0.0)
        t_it = (time.perf_counter() - t0) / (it + 1)
    n_newton = gpu['newton_steps']
    cpu_round = t_samp + t_bc + max(1, n_newton) * t_it
    return {"workload": "L=99 q=4 round: 16384 walkers x 64 sweeps, bicounts, quasi-Newton",
            "gpu_round_s": gpu['wall_s'], "gpu_newton_steps": n_newton,
            "gpu_mcmc_s": gpu['mcmc_s'], "gpu_newton_s": gpu['newton_s'],
            "cpu_round_s_est": cpu_round, "cpu_sampler_s": t_samp, "cpu_sampler_threads": nthr,
            "cpu_bicounts_s": t_bc, "cpu_newton_iter_s": t_it,
            "speedup_round": cpu_round / gpu['wall_s'],
            "note": "CPU round = sampler + numpy bicounts + GPU's Newton iteration count x "
                    "measured numpy iteration time (4 iterations timed)"}


def result_line(out):
    """The one line of standard output: `out` without the runs' lists of rounds, which
    made it longer (16 KB for 64 rounds) than what is kept of a run's output.  Those
    go to standard error."""
    short = dict(out)
    for key in ('round', 'hiv_reference_run'):
        if key in short:
            print(f"{key}, rounds: {json.dumps(short[key]['rounds'])}", file=sys.stderr, flush=True)
            short[key] = dict(short[key], rounds=len(short[key]['rounds']))
    return json.dumps(short)


def copy_calibration(mib):
    """Plain device-to-device copies of a known size: a profiler run that
    also covers them turns FETCH_SIZE / WRITE_SIZE counts into bytes."""
    from mi3gpu._lib import lib, check
    import ctypes
    ctx = ctypes.c_void_p()
    check(None, lib().mi3_create(0, 8, 4, 512, 1, 0, ctypes.byref(ctx)))
    nbytes = mib << 20
    for name in (b'copy src', b'copy dst'):
        check(ctx, lib().mi3_buf_alloc(ctx, name, nbytes))
    check(ctx, lib().mi3_buf_fill_u32(ctx, b'copy src', 0x01020304))
    for _ in range(3):
        check(ctx, lib().mi3_buf_copy(ctx, b'copy dst', b'copy src', nbytes))
    check(ctx, lib().mi3_synchronize(ctx))
    lib().mi3_destroy(ctx)


def achievable_hbm(mib=4096, reps=10):
    """HBM bandwidth a plain copy reaches (read + write bytes over wall time
    between synchronisations), GB/s: the better of the runtime's
    device-to-device copy and the library's streaming-copy kernel."""
    from mi3gpu._lib import lib, check
    import ctypes
    ctx = ctypes.c_void_p()
    check(None, lib().mi3_create(0, 8, 4, 512, 1, 0, ctypes.byref(ctx)))
    nbytes = mib << 20
    for name in (b'copy src', b'copy dst'):
        check(ctx, lib().mi3_buf_alloc(ctx, name, nbytes))
    check(ctx, lib().mi3_buf_fill_u32(ctx, b'copy src', 0x01020304))
    rates = {}
    runs = (('hipMemcpy device-to-device copy', 2,
             lambda: lib().mi3_buf_copy(ctx, b'copy dst', b'copy src', nbytes)),
            ('streaming-copy kernel', 2,
             lambda: lib().mi3_stream_copy(ctx, b'copy dst', b'copy src', nbytes)),
            ('streaming-read kernel', 1,
             lambda: lib().mi3_stream_read(ctx, b'copy src', nbytes, b'copy dst')))
    for kind, passes, fn in runs:
        check(ctx, fn())
        check(ctx, lib().mi3_synchronize(ctx))
        t0 = time.perf_counter()
        for _ in range(reps):
            check(ctx, fn())
        check(ctx, lib().mi3_synchronize(ctx))
        rates[kind] = passes * nbytes * reps / (time.perf_counter() - t0) / 1e9
    lib().mi3_destroy(ctx)
    kind = max(rates, key=rates.get)
    return rates[kind], f"{kind} of {mib} MiB x {reps}, bytes moved over wall time", rates


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument('--gpus', type=int, default=1)
    ap.add_argument('--steps', type=int, default=20)
    ap.add_argument('--warmup', type=int, default=3)
    ap.add_argument('--walkers', type=int, default=2 ** 18)
    ap.add_argument('--sweeps-per-step', type=int, default=8)
    ap.add_argument('--wgsize', type=int, default=512,
                    help="walkers per work-group of the sweep (128, 256, 512)")
    ap.add_argument('--no-cpu', action='store_true', help="skip the CPU baseline")
    ap.add_argument('--ess-sweeps', type=int, default=128,
                    help="traced sweeps for energy-ESS (0 = skip)")
    ap.add_argument('--target-sweeps', type=int, default=256,
                    help="sweeps to sample the 2^20 target sequences")
    ap.add_argument('--rounds', type=int, default=2,
                    help="Mi3 inference rounds to time (0 = skip)")
    ap.add_argument('--round-equiltime', default='8',
                    help="equiltime of the timed rounds (launches of 16 sweeps, or 'auto')")
    ap.add_argument('--round-nsteps', type=int, default=0,
                    help="nsteps of the timed rounds (default 16*L)")
    ap.add_argument('--hiv-rounds', type=int, default=64,
                    help="rounds of the reference's HIV example (pbs.sh settings, 64 in the "
                         "reference) compared with its published convergence; it gives the "
                         "s per round at fixed SSR (0 skips it)")
    ap.add_argument('--no-config1', action='store_true',
                    help="skip the L=99 q=4 round on the GPU and its CPU reference path")
    ap.add_argument('--kernels', action='store_true',
                    help="also time bicounts and energies standalone on 2^20 sequences, "
                         "and one quasi-Newton iteration's kernels on 2^18")
    ap.add_argument('--batch-rounds', type=int, default=0,
                    help="also time the batched uneven-models workload (rounds)")
    ap.add_argument('--made', action='store_true',
                    help="also measure the learned proposal (MADE mixed 1:8 with sweeps, "
                         "2^16 walkers) against the plain sweep")
    ap.add_argument('--made-train-steps', type=int, default=1500)
    ap.add_argument('--copy-calibration', type=int, default=0, metavar='MIB',
                    help="also run 3 device-to-device copies of MIB MiB (the reference "
                         "kernel that scales HBM byte counters)")
    a = ap.parse_args()
    if a.gpus != 1:
        print(f"bench.py measures one GPU; --gpus {a.gpus} is not supported: this engine "
              "runs on a single device (the sampler would shard by walker, with one "
              "all-reduce of the int32 bicounts per round)", file=sys.stderr)
        sys.exit(2)

    from mi3gpu.mcmcGPU import MCMCGPU
    L, q, N = 232, 21, a.walkers
    nsteps = a.sweeps_per_step * L
    J = production_model(L, q, seed=1)
    s0 = np.random.default_rng(2).integers(0, q, size=(N, L)).astype('<u1')
    with tempfile.TemporaryDirectory() as d:
        g = MCMCGPU((0, 0, None, None), L, q, N, a.wgsize, Path(d), 1024, 2, profile=True)
        g.initMCMC(nsteps, 0, 2 ** 63)
        g.setBuf('J', J)
        g.setBuf('seq main', s0)
        for _ in range(a.warmup):
            g.runMCMC()
        g.wait()
        g.profile_reset()
        t0 = time.perf_counter()
        for _ in range(a.steps):
            g.runMCMC()
        g.wait()
        dt = time.perf_counter() - t0
        kms, kcnt = g.kernel_ms('mcmc')
        # the same launches' coupling staging alone (same sites, chunks and
        # launch shape; walker state untouched)
        from mi3gpu._lib import lib, check
        for _ in range(3):
            check(g._ctx, lib().mi3_stage_probe(g._ctx, 1))
            check(g._ctx, lib().mi3_stage_probe(g._ctx, 2))
        g.wait()
        p1_ms, _ = g.kernel_ms('stageProbe')
        p2_ms, _ = g.kernel_ms('stageProbe2')
        # energies of the final ensemble (sanity)
        g.calcEnergies('main')
        E = g.getBuf('E main').read()

    if a.copy_calibration > 0:
        copy_calibration(a.copy_calibration)
    hbm_copy, hbm_kind, hbm_rates = achievable_hbm()

    su_per_step = N * nsteps
    value = su_per_step * a.steps / dt
    alg_bytes = su_per_step * (L + 1)
    achieved = alg_bytes / (kms * 1e-3) / 1e9
    key = (L, q, N, a.sweeps_per_step, a.wgsize)
    # bytes every work-group copies from L2 into LDS per launch: the padded
    # coupling chunks of each step's site
    chunk_bytes = _pf_class(q) * 512 * 16
    nchunk = (L + 31) // 32
    wgs = N // a.wgsize
    stage_bytes = wgs * nsteps * nchunk * chunk_bytes
    onchip = {
        "binding": "on-chip: VALU issue (gathers) and the L2->LDS coupling staging; HBM "
                   "traffic is 0.12 of the algorithmic bytes",
        "staging_bytes_per_launch": stage_bytes,
        "staging_TBps": stage_bytes / (kms * 1e-3) / 1e12,
        "staging_alone_ms": p1_ms,
        "staging_alone_TBps": stage_bytes / (p1_ms * 1e-3) / 1e12,
        "staging_alone_2inflight_ms": p2_ms,
        "staging_alone_2inflight_TBps": stage_bytes / (p2_ms * 1e-3) / 1e12,
        "sweep_over_staging_alone": kms / p1_ms,
        "lds_gather_bytes_per_launch": su_per_step * 8 * (L - 1),
        "lds_gather_TBps": su_per_step * 8 * (L - 1) / (kms * 1e-3) / 1e12,
        "valu_busy_profiled": MEASURED_VALU_BUSY.get(key),
    }
    out = {
        "metric": METRIC,
        "value": value,
        "unit": "site-updates/s",
        "n_gpus": 1,
        "steps": a.steps,
        "warmup": a.warmup,
        "ms_per_step": dt / a.steps * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": "plain Mi3 Metropolis sweep, L=232 q=21, 2^18 walkers, random "
                               "Potts model h~N(0,1) J~N(0,0.05) zero-sum gauge folded "
                               "fieldless float32",
                   "L": L, "q": q, "walkers": N, "sweeps_per_step": a.sweeps_per_step,
                   "walkers_per_workgroup": a.wgsize,
                   "mean_energy_after": float(np.mean(E))},
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS, "traffic": MEASURED_TRAFFIC.get(key),
                     "kernel": "k_sweep", "kernel_ms": kms, "launches": kcnt,
                     "alg_bytes_per_launch": alg_bytes,
                     "achievable": hbm_copy, "frac_of_achievable": achieved / hbm_copy,
                     "achievable_kind": hbm_kind,
                     "achievable_all": hbm_rates,
                     "onchip": onchip},
    }
    if a.ess_sweeps > 0 or a.rounds > 0 or a.made:
        tseqs, target = sample_target(J, L, q, 2 ** 20, a.target_sweeps, 4, a.wgsize)
        if a.ess_sweeps > 0:
            out["energy_ess"] = measure_ess(J, tseqs[:N], L, q, a.ess_sweeps, 5, a.wgsize)
        if a.made:
            out["learned_proposal"] = measure_made(J, tseqs, L, q,
                                                   train_steps=a.made_train_steps)
        del tseqs
        if a.rounds > 0:
            out["round"] = measure_rounds(target, L, q, N, a.rounds, 6, a.round_equiltime,
                                          a.round_nsteps or None)
    if a.kernels:
        out["kernels"] = measure_kernels()
        out["newton_kernels"] = measure_newton_kernels()
    if a.hiv_rounds > 0:
        hiv = measure_hiv(a.hiv_rounds)
        out["hiv_reference_run"] = hiv
        # the third metric: wall time of the first round within twice the
        # SSR floor, on the reference's own published run
        fx = hiv["fixed_ssr"]
        out["s_per_round_at_fixed_ssr"] = None if fx is None else {
            "value": fx["s"], "unit": "s/round",
            "s_without_seq_write": fx["s_without_seq_write"], "round": fx["round"], "ssr": fx["ssr"],
            "ssr_floor": hiv["ssr_floor"], "cumulative_s": fx["cumulative_s"],
            "workload": hiv["workload"]}
    if not a.no_config1 and not a.no_cpu:
        out["config1_round"] = measure_config1()
    if a.batch_rounds > 0:
        out["batch"] = measure_batch(a.batch_rounds)
    if not a.no_cpu:
        out["cpu_baseline"] = cpu_baseline(J, L, q, seed=3)
    print(result_line(out), flush=True)


if __name__ == '__main__':
    main()
