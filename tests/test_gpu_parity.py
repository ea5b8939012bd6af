"""GPU parity of the HIP engine against the FP64 oracle (same variates).

Bars (per-move energies in kJ/mol; 1e-4 kcal/mol = 4.184e-4 kJ/mol):
* trial centres, poses, included-group sets, slots: bit-exact;
* trial energies: |E_gpu - E_fp64| <= 4.184e-4 kJ/mol when |E| <= 200 kJ/mol
  (every trial with a Boltzmann weight above e^-80); beyond, where strongly
  repulsive LJ terms carry FP32 relative error, 1e-5 relative;
* accept/reject decisions and picks: identical on >= 99.99% of groups;
* final state after a lock-step replay: bit-identical.
"""

import numpy as np
import pytest

from oracle import oracle as O
from pygcmc_amd.engine import Engine

from . import systems

pytestmark = pytest.mark.gpu

KCAL = 4.184e-4


def e_tol(e):
    e = np.abs(e)
    return np.where(e <= 200.0, KCAL, np.maximum(KCAL, 1e-5 * e))


def band_report(e_ref, err):
    out = []
    for lo, hi in ((0, 50), (50, 200), (200, 1000), (1000, np.inf)):
        m = (np.abs(e_ref) > lo) & (np.abs(e_ref) <= hi) if lo else np.abs(e_ref) <= hi
        if m.any():
            out.append(f'|E|<={hi:g}: n={m.sum()} max {err[m].max():.2e} rms {np.sqrt((err[m] ** 2).mean()):.2e}')
    return '; '.join(out)


def test_eval_poses_matches_fp64():
    s = systems.populated_water()
    eng = Engine()
    eng.add_system(s)
    eng.upload()
    c, p = systems.random_poses(s, 0, 1024, seed=7)
    E, N, H = eng.eval_poses(0, 0, c, p)
    ref = np.array([O.energy_pose(s, 0, c[i], p[i]) for i in range(len(c))], dtype=object)
    e = ref[:, 0].astype(np.float64)
    assert np.array_equal(ref[:, 1].astype(np.int64), N.astype(np.int64))
    assert np.array_equal(ref[:, 2].astype(np.uint64), H.astype(np.uint64))
    err = np.abs(e - E)
    print('eval_poses (kJ/mol):', band_report(e, err))
    assert (err <= e_tol(e)).all(), (err.max(), e[err.argmax()])
    eng.close()


@pytest.mark.parametrize('n', [1, 5, 1023, 1024, 1025, 16000])
def test_eval_poses_by_number(n):
    """Poses shared by four waves (fewer than 1,024) or one wave's, one call's in
    pinned memory or (16,000: above 1 MiB) in device memory: every form gives the
    groups of a pose exactly and its energy to the order of an FP64 sum."""
    s = systems.populated_water()
    eng = Engine()
    eng.add_system(s)
    eng.upload()
    c, p = systems.random_poses(s, 0, 1024, seed=9)
    parts = [eng.eval_poses(0, 0, c[i:i + 64], p[i:i + 64]) for i in range(0, 1024, 64)]
    ref = [np.concatenate([x[k] for x in parts]) for k in range(3)]
    q = np.random.default_rng(n).integers(0, 1024, n)
    E, N, H = eng.eval_poses(0, 0, c[q], p[q])
    assert np.array_equal(N, ref[1][q]) and np.array_equal(H, ref[2][q])
    # at most some 1,000 FP64 terms, the largest not above 100 times the sum of
    # a pose that matters: 1e-10 of the energy, or of 1 kJ/mol
    assert (np.abs(E - ref[0][q]) <= 1e-10 * np.maximum(np.abs(ref[0][q]), 1.0)).all()
    eng.close()


@pytest.mark.parametrize('terms', ['fp32', 'ewald'])
def test_eval_poses_by_number_fp32_terms(terms):
    """The same for FP32 pair terms, plain and Ewald: a pair's term is the same in
    either form, so energies agree to the order of an FP64 sum."""
    s = systems.populated_water()
    eng = Engine(fp32_coulomb=1 if terms == 'fp32' else 0)
    eng.add_system(s)
    if terms == 'ewald':
        eng.set_ewald(0, 0.34, 1.0)
    eng.upload()
    c, p = systems.random_poses(s, 0, 1500, seed=10)
    E, N, H = eng.eval_poses(0, 0, c, p)
    for i in range(0, 1500, 500):
        e, n, h = eng.eval_poses(0, 0, c[i:i + 500], p[i:i + 500])
        assert np.array_equal(N[i:i + 500], n) and np.array_equal(H[i:i + 500], h)
        assert (np.abs(E[i:i + 500] - e) <= 1e-10 * np.maximum(np.abs(e), 1.0)).all()
    eng.close()


@pytest.mark.parametrize('excluding', [False, True])
def test_eval_poses_in_chunks(excluding):
    """More poses than go to the GPU at once (65,536), with and without excluded
    molecules, then a small call in the same buffers."""
    s = systems.populated_water()
    eng = Engine()
    eng.add_system(s)
    eng.upload()
    c, p = systems.random_poses(s, 0, 256, seed=12)
    n = 65536 + 321
    rng = np.random.default_rng(3)
    q = rng.integers(0, 256, n)
    first = int(s['frag'][0]['startRes'])
    ex = np.where(np.arange(256) % 3 == 0, -1, first + np.arange(256) % int(s['frag'][0]['totalNum'])).astype(np.int32)
    pick = (lambda i: ex[i]) if excluding else (lambda i: None)
    parts = [eng.eval_poses(0, 0, c[i:i + 64], p[i:i + 64], pick(slice(i, i + 64))) for i in range(0, 256, 64)]
    ref = [np.concatenate([x[k] for x in parts]) for k in range(3)]
    for i in (q, q[-70:]):
        E, N, H = eng.eval_poses(0, 0, c[i], p[i], pick(i))
        assert np.array_equal(N, ref[1][i]) and np.array_equal(H, ref[2][i])
        assert (np.abs(E - ref[0][i]) <= 1e-10 * np.maximum(np.abs(ref[0][i]), 1.0)).all()
    eng.close()


def test_water_fixture_on_gpu():
    """The reference's 3-water insertion (test/water/3water.pdb) on the GPU."""
    for ch, lj, key in ((True, False, 'expected_coulomb_kj'), (False, True, 'expected_lj_kj')):
        s, c, p, fx = systems.water3_system(ch, lj)
        eng = Engine()
        eng.add_system(s)
        eng.upload()
        E, N, H = eng.eval_poses(0, 0, c[None], p[None])
        eng.close()
        ref = O.energy_pose(s, 0, c, p)[0]
        assert abs(E[0] - ref) <= KCAL and N[0] == 2
        assert abs(E[0] - fx[key]) < 3e-4


def _lockstep(sysd, nsteps, mode='plain', max_k=None, wg_size=0):
    max_k = max_k or int(sysd['frag']['confBias'].max())
    gpu_sys = systems.copy(sysd)
    eng = Engine(wg_size=wg_size)
    eng.add_system(gpu_sys)
    eng.upload()
    eng.set_trace(0, nsteps, max_k)
    eng.run(nsteps, mode)
    gt = eng.get_trace(0)
    eng.download(0)
    st = eng.stats(0)
    eng.close()
    ref = systems.copy(sysd)
    ot = O.new_trace(nsteps, max_k)
    O.run(ref, first=0, nsteps=nsteps, trace=ot, follow=gt)
    return gt, ot, gpu_sys, ref, st


def _compare(gt, ot, gpu_sys, ref):
    assert np.array_equal(gt['k'], ot['k'])
    kmask = np.arange(gt['centre'].shape[1])[None, :] < gt['k'][:, None]
    assert np.array_equal(gt['centre'][kmask], ot['centre'][kmask])
    assert np.array_equal(gt['posehash'][kmask], ot['posehash'][kmask])
    assert np.array_equal(gt['ninc'][kmask], ot['ninc'][kmask])
    assert np.array_equal(gt['inchash'][kmask], ot['inchash'][kmask])
    eg, eo = gt['e'][kmask], ot['e'][kmask]
    err = np.abs(eg - eo)
    print('trial energies (kJ/mol):', band_report(eo, err))
    assert (err <= e_tol(eo)).all(), (err.max(), eo.ravel()[err.argmax()])
    gmask = np.arange(gt['gpick'].shape[1])[None, :] < gt['ngroups'][:, None]
    ng = int(gmask.sum())
    mism = int((gt['gpick'][gmask] != ot['gpick'][gmask]).sum() +
               (gt['gacc'][gmask] != ot['gacc'][gmask]).sum())
    assert mism <= max(0, int(1e-4 * ng)), (mism, ng)
    assert np.array_equal(gt['naccept'], ot['naccept']) or mism > 0
    # lock-step replay leaves bit-identical states
    assert np.array_equal(gpu_sys['frag']['totalNum'], ref['frag']['totalNum'])
    assert np.array_equal(gpu_sys['res']['position'].view(np.uint32), ref['res']['position'].view(np.uint32))
    assert np.array_equal(gpu_sys['atoms'].view(np.uint8), ref['atoms'].view(np.uint8))
    return float(err.max()), ng, mism


def test_lockstep_water_plain():
    s = systems.water(nsteps=600, conf=3)
    gt, ot, g, r, st = _lockstep(s, 600, 'plain')
    err, ng, mism = _compare(gt, ot, g, r)
    print(f'water plain: max |dE| {err:.3e} kJ/mol over {ng} groups, {mism} mismatches, '
          f'N={g["frag"]["totalNum"]}')
    assert g['frag']['totalNum'][0] > 0


def test_lockstep_water_batched():
    s = systems.water(nsteps=600, conf=3)
    gt, ot, g, r, st = _lockstep(s, 600, 'batched')
    err, ng, mism = _compare(gt, ot, g, r)
    print(f'water batched: max |dE| {err:.3e}, {ng} groups, {mism} mismatches')


@pytest.mark.parametrize('wg_size', [256, 512, 1024])
def test_lockstep_multi_fragment(wg_size):
    s = systems.multi(nsteps=400)
    gt, ot, g, r, st = _lockstep(s, 400, 'batched', wg_size=wg_size)
    err, ng, mism = _compare(gt, ot, g, r)
    print(f'multi batched: max |dE| {err:.3e}, {ng} groups, {mism} mismatches, N={g["frag"]["totalNum"]}')


@pytest.mark.parametrize('dx', [-1.5, 2.0, 3.0])
def test_lockstep_translation_steps(dx):
    """Translations whose two centres are served by one scan (up to 2 A), and by
    two (wider or negative steps)."""
    s = systems.multi(nsteps=600)
    s['info']['grid_dx'] = dx
    gt, ot, g, r, st = _lockstep(s, 600, 'batched')
    err, ng, mism = _compare(gt, ot, g, r)
    trn = st['attempts'][:, 2].sum()
    print(f'grid_dx {dx}: max |dE| {err:.3e}, {ng} groups, {mism} mismatches, {trn} translations')
    assert trn > 50 and (gt['k'][s['moves'][:600] % 4 == 2] > 0).sum() > 20


@pytest.mark.parametrize('mode', ['plain', 'batched', 'graph'])
def test_evaluation_time_by_phase(mode):
    """Every phase of the evaluations has its time, whether four waves share a
    trial or one has it (fewer and more than 100 trials per move)."""
    for conf in (4, 130):
        s = systems.water(nsteps=300, conf=conf)
        eng = Engine()
        eng.add_system(s)
        eng.upload()
        assert not any(eng.eval_sub_seconds(0).values())
        ms = eng.run(300, mode)
        t = eng.eval_sub_seconds(0)
        n = eng.counters(0)['evals']
        print(mode, conf, n, {k: f'{1e9 * v / n:.0f} ns per evaluation' for k, v in t.items()})
        assert all(v > 0.0 for v in t.values())
        assert sum(t.values()) < 1e-3 * ms * 256 * 12   # all waves that fit on the GPU, all the time
        eng.close()


@pytest.mark.parametrize('wg_size', [256, 1024])
def test_plain_batched_graph_identical(wg_size):
    s = systems.multi(nsteps=300, seed=11)
    outs = []
    for mode in ('plain', 'batched', 'graph'):
        g = systems.copy(s)
        eng = Engine(wg_size=wg_size)
        eng.add_system(g)
        eng.upload()
        eng.set_trace(0, 300, int(s['frag']['confBias'].max()))
        for _ in range(3):
            eng.run(100, mode)
        tr = eng.get_trace(0)
        eng.download(0)
        st = eng.stats(0)
        eng.close()
        outs.append((tr, g, st))
    for tr, g, st in outs[1:]:
        assert np.array_equal(tr['e'].view(np.uint64), outs[0][0]['e'].view(np.uint64))
        assert np.array_equal(tr['gacc'], outs[0][0]['gacc'])
        assert np.array_equal(g['atoms'].view(np.uint8), outs[0][1]['atoms'].view(np.uint8))
        assert st['energy'] == outs[0][2]['energy']


def test_pair_rows_in_lds_identical():
    """The pair table held in LDS (copied with global_load_lds) or read
    from global memory: the same values, so bit-identical energies and
    chains, in the batched and plain forms."""
    s = systems.multi(nsteps=300, seed=13)
    outs = []
    for pair_lds in (-1, 0):
        for mode in ('batched', 'plain'):
            g = systems.copy(s)
            eng = Engine(pair_lds=pair_lds)
            eng.add_system(g)
            eng.upload()
            eng.set_trace(0, 300, int(s['frag']['confBias'].max()))
            eng.run(300, mode)
            tr = eng.get_trace(0)
            eng.download(0)
            eng.close()
            outs.append((tr, g))
    for tr, g in outs[1:]:
        assert np.array_equal(tr['e'].view(np.uint64), outs[0][0]['e'].view(np.uint64))
        assert np.array_equal(g['atoms'].view(np.uint8), outs[0][1]['atoms'].view(np.uint8))


def test_replicas_match_single_runs():
    """Uneven replicas in one persistent kernel give the same chains as
    each system run alone."""
    sizes = [(1000, 30.0, 21), (2500, 45.0, 22), (1600, 38.0, 23), (1200, 33.0, 24), (900, 28.0, 25),
             (2000, 42.0, 26), (1500, 36.0, 27), (1800, 40.0, 28), (1100, 31.0, 29), (2200, 44.0, 30)]
    base = [systems.multi(nsteps=200, n_fixed=n, box=b, seed=sd) for n, b, sd in sizes]
    eng = Engine()
    batch = [systems.copy(s) for s in base]
    for b in batch:
        eng.add_system(b)
    eng.upload()
    eng.run(200, 'batched')
    for r in range(len(batch)):
        eng.download(r)
    eng.close()
    for s, b in zip(base, batch):
        one = systems.copy(s)
        e1 = Engine()
        e1.add_system(one)
        e1.upload()
        e1.run(200, 'plain')
        e1.download(0)
        e1.close()
        assert np.array_equal(one['atoms'].view(np.uint8), b['atoms'].view(np.uint8))
        assert np.array_equal(one['frag']['totalNum'], b['frag']['totalNum'])


def test_rungcmc_dropin_matches_oracle():
    """pygcmc_amd.gpu.runGCMC: same arrays, same in-place contract as gcmc.gpu.runGCMC."""
    from pygcmc_amd import gpu
    s = systems.water(nsteps=400, conf=2)
    g = systems.copy(s)
    gpu.runGCMC(g['info'], g['frag'], g['res'], g['atoms'], g['grid'], g['ff'], g['moves'])
    ref = systems.copy(s)
    O.run(ref)
    assert np.array_equal(g['frag']['totalNum'], ref['frag']['totalNum'])
    assert np.array_equal(g['atoms'].view(np.uint8), ref['atoms'].view(np.uint8))
    assert np.array_equal(g['res'].view(np.uint8), ref['res'].view(np.uint8))


def test_lockstep_bench_replica():
    """First replica of the 64-system benchmark (uneven sizes; 8 fragments +
    water, full confBias): lock-step against the FP64 oracle at the bars."""
    from pygcmc_amd import synth
    sizes = synth.replica_sizes(64)
    s = synth.replica_system(0, int(sizes[0]), mcsteps=300)
    gt, ot, g, r, st = _lockstep(s, 300, 'batched')
    err, ng, mism = _compare(gt, ot, g, r)
    print(f'bench replica 0 ({int(sizes[0])} fixed atoms): max |dE| {err:.3e}, {ng} groups, {mism} mismatches')


def test_rejects_group_ids_beyond_cell_record_word():
    # a mobile group's cell record carries its id in 24 bits: larger systems
    # are refused at add_system, before any array is read
    from pygcmc_amd import synth
    s = synth.water_sphere(mcsteps=10, conf=3)
    s['info'] = s['info'].copy()
    s['info']['totalResNum'] = 1 << 24
    eng = Engine()
    try:
        with pytest.raises(RuntimeError, match='totalResNum'):
            eng.add_system(s)
    finally:
        eng.close()


def test_snapshot_restore_reruns_identical_chain():
    """restore() returns every system to the snapshot: a rerun gives the same
    trace, statistics, counters and final arrays, in the batched and graph
    forms, and after a plain run too."""
    base = [systems.multi(nsteps=150, seed=31), systems.water(nsteps=150, conf=3)]
    batch = [systems.copy(s) for s in base]
    eng = Engine()
    for b in batch:
        eng.add_system(b)
    eng.upload()
    eng.snapshot()
    runs = []
    for mode in ('batched', 'graph', 'plain', 'batched'):
        eng.restore()
        assert [eng.step(r) for r in range(2)] == [0, 0]
        eng.run(150, mode)
        out = []
        for r in range(2):
            st = eng.stats(r)
            g = systems.copy(base[r])
            eng.download(r, g)
            out.append((st['energy'], st['accepts'].copy(), eng.counters(r), g['atoms'].view(np.uint8).copy(),
                        g['frag']['totalNum'].copy()))
        runs.append(out)
    eng.close()
    for out in runs[1:]:
        for (e, acc, cnt, atoms, n), (e0, acc0, cnt0, atoms0, n0) in zip(out, runs[0]):
            assert e == e0 and np.array_equal(acc, acc0) and cnt == cnt0
            assert np.array_equal(atoms, atoms0) and np.array_equal(n, n0)
    # the chain moved: something was accepted
    assert runs[0][0][1].sum() > 0


def test_xcd_assignment_never_changes_chains():
    """Systems assigned to XCDs round-robin, by estimated work, by the work
    measured in the previous run (the second run of a snapshot), or by the
    exchanges tried on later runs of the same steps: the same final states."""
    base = [systems.multi(nsteps=200, n_fixed=n, box=b, seed=sd, conf_scale=0.2)
            for n, b, sd in ((900, 28.0, 41), (2400, 44.0, 42), (1500, 36.0, 43), (1200, 33.0, 44),
                             (2000, 42.0, 45), (1000, 30.0, 46), (1800, 40.0, 47), (1300, 34.0, 48),
                             (2200, 43.0, 49), (1100, 31.0, 50))]
    finals = []
    for rr in (1, 0):
        eng = Engine(xcd_round_robin=rr)
        gs = [systems.copy(b) for b in base]
        for g in gs:
            eng.add_system(g)
        eng.upload()
        eng.snapshot()
        # the second run is balanced by the first's measured work; the third
        # to fifth try exchanges of two systems between XCDs
        for _ in range(5):
            eng.restore()
            eng.run(200, 'batched')
            out = []
            for r in range(len(gs)):
                g = systems.copy(base[r])
                eng.download(r, g)
                out.append(g['atoms'].view(np.uint8).copy())
            finals.append(out)
        eng.close()
    for out in finals[1:]:
        for a, b in zip(out, finals[0]):
            assert np.array_equal(a, b)


@pytest.mark.parametrize('conf', [63, 64, 65, 96, 97, 130, 256, 300])
def test_selection_by_number_of_trials(conf):
    """Lock-step with the oracle at the trial counts where the selection changes
    its form (64 trials in registers, above that batches of 64 groups): word
    and wave boundaries of the member masks, moves of more groups than one
    batch holds, acceptances inside a batch."""
    from pygcmc_amd import synth
    s = synth.water_sphere(mcsteps=40, conf=conf, n_fixed=3000, radius=25.0, box=100.0)
    gt, ot, g, r, st = _lockstep(s, 40, 'batched', max_k=conf)
    _compare(gt, ot, g, r)
    print('groups', gt['ngroups'].max(), 'accepted', gt['naccept'].sum())
    assert gt['naccept'].sum() > 0
    assert conf < 256 or gt['ngroups'].max() > 64
