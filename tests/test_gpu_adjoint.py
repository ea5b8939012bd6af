"""The HIP adjoint (pygcmc_amd.adjoint) against the FP64 oracle gradient and
central finite differences of the FP64 energy (h = 1e-4).

Bars: energies as the MC path (4.184e-4 kJ/mol for |E| <= 200 kJ/mol);
per-pose coordinate gradients and loss gradients in the per-type parameters
within 1e-4 relative (2-norm over the pose's atoms / over the types).
"""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from pygcmc_amd import adjoint
from pygcmc_amd.engine import Engine

from . import systems

pytestmark = pytest.mark.gpu

KCAL = 4.184e-4


def _setup(n_per_species=24, seed=41):
    s = systems.multi(nsteps=10, n_fixed=6000, box=60.0)
    eng = Engine()
    eng.add_system(s)
    eng.upload()
    eps, rmin = adjoint.type_parameters(s)
    poses = {}
    T = int(s['info'][0]['fragTypeNum'])
    for spi in range(T):
        poses[spi] = systems.moderate_poses(s, spi, n_per_species, seed=seed + spi)
    return s, eng, eps, rmin, poses


@pytest.fixture(scope='module')
def case():
    s, eng, eps, rmin, poses = _setup()
    yield s, eng, eps, rmin, poses
    eng.close()


def _gpu(eng, spi, c, p, eps, rmin, dq=None):
    ct = torch.tensor(c, device='cuda')
    pt = torch.tensor(p, device='cuda', requires_grad=True)
    e = eps.clone().requires_grad_(True)
    r = rmin.clone().requires_grad_(True)
    q = (torch.zeros_like(eps) if dq is None else dq.clone()).requires_grad_(True)
    E = adjoint.pose_energy(eng, 0, spi, ct, pt, e, r, q)
    return E, pt, e, r, q


def test_adjoint_energy_matches_fp64_and_mc_path(case):
    """Energies against the FP64 oracle with the same per-type parameters
    (1e-4 kcal/mol), and against the MC path's energies, whose pair table
    rounds (sigma, epsilon) once per pair instead of once per type: within
    2e-6 of the sum of |pair terms| scale, bounded here by 5e-3 kJ/mol."""
    s, eng, eps, rmin, poses = case
    e64p, r64p = eps.double().cpu().numpy(), rmin.double().cpu().numpy()
    for spi, (c, p) in poses.items():
        E, *_ = _gpu(eng, spi, c, p, eps, rmin)
        e_mc, n, _ = eng.eval_poses(0, spi, c, p)
        e64 = np.array([O.adjoint(s, spi, c[i], p[i], e64p, r64p)[0] for i in range(len(c))])
        Eg = E.detach().cpu().numpy()
        assert np.abs(Eg - e64).max() <= KCAL, (spi, np.abs(Eg - e64).max())
        assert np.abs(Eg - e_mc).max() <= 5e-3, (spi, np.abs(Eg - e_mc).max())


def test_adjoint_pose_gradients_match_fp64(case):
    s, eng, eps, rmin, poses = case
    e64, r64 = eps.double().cpu().numpy(), rmin.double().cpu().numpy()
    worst = 0.0
    for spi, (c, p) in poses.items():
        E, pt, *_ = _gpu(eng, spi, c, p, eps, rmin)
        E.sum().backward()
        g = pt.grad.cpu().numpy()
        for i in range(len(c)):
            gref = O.adjoint(s, spi, c[i], p[i], e64, r64)[1]
            rel = np.linalg.norm(g[i] - gref) / max(np.linalg.norm(gref), 1e-3)
            worst = max(worst, rel)
    print(f'pose gradient: worst relative error vs FP64 {worst:.2e}')
    assert worst <= 1e-4


def test_adjoint_type_gradients_match_fp64(case):
    s, eng, eps, rmin, poses = case
    e64, r64 = eps.double().cpu().numpy(), rmin.double().cpu().numpy()
    rng = np.random.default_rng(3)
    dq = torch.tensor(rng.normal(0, 0.02, len(e64)), dtype=torch.float32, device='cuda')
    dq64 = dq.double().cpu().numpy()
    for spi, (c, p) in poses.items():
        w = rng.normal(size=len(c))
        E, pt, e, r, q = _gpu(eng, spi, c, p, eps, rmin, dq)
        (E * torch.tensor(w, device='cuda')).sum().backward()
        ref = np.zeros((3, len(e64)))
        for i in range(len(c)):
            _, _, gq, ge, gr = O.adjoint(s, spi, c[i], p[i], e64, r64, dq64)
            ref += w[i] * np.stack([gq, ge, gr])
        got = np.stack([q.grad.cpu().numpy(), e.grad.cpu().numpy(), r.grad.cpu().numpy()])
        for k, name in enumerate(('dq', 'eps', 'rmin')):
            rel = np.linalg.norm(got[k] - ref[k]) / max(np.linalg.norm(ref[k]), 1e-3)
            print(f'species {spi} {name}: relative error {rel:.2e}')
            assert rel <= 1e-4, (spi, name, rel)


def test_adjoint_matches_finite_differences(case):
    """GPU gradients against central differences (h = 1e-4) of the FP64 energy."""
    s, eng, eps, rmin, poses = case
    e64, r64 = eps.double().cpu().numpy(), rmin.double().cpu().numpy()
    for spi in (0, 4, 8):
        c, p = poses[spi]
        c, p = c[:2], p[:2]
        E, pt, e, r, q = _gpu(eng, spi, c[:1], p[:1], eps, rmin)
        E.sum().backward()
        fd = systems.fd_pose_gradient(s, spi, c[0], p[0], e64, r64)
        g = pt.grad.cpu().numpy()[0]
        assert np.linalg.norm(g - fd) <= 1e-4 * np.linalg.norm(fd)
        for which, got in (('q', q.grad), ('eps', e.grad), ('rmin', r.grad)):
            got = got.cpu().numpy()
            for t in np.argsort(-np.abs(got))[:4]:
                d = systems.fd_type_gradient(s, spi, c[0], p[0], e64, r64, which, int(t))
                assert abs(got[t] - d) <= 1e-4 * max(abs(d), 1e-2), (spi, which, t, got[t], d)


def test_adjoint_rejects_bad_shapes(case):
    s, eng, eps, rmin, poses = case
    c, p = poses[0]
    with pytest.raises(ValueError):
        adjoint.pose_energy(eng, 0, 0, torch.tensor(c, device='cuda'),
                            torch.tensor(p[:, :-1], device='cuda'), eps, rmin)
    with pytest.raises(TypeError):
        adjoint.pose_energy(eng, 0, 0, torch.tensor(c), torch.tensor(p), eps, rmin)


@pytest.mark.parametrize('n', [1, 2047, 2048, 2049])
def test_adjoint_by_number_of_poses(case, n):
    """Poses shared by four waves (fewer than 2,048) or one wave's: energies to the
    order of an FP64 sum, coordinate gradients within this file's bar."""
    s, eng, eps, rmin, poses = case
    c, p = poses[2]
    E0, pt0, *_ = _gpu(eng, 2, c, p, eps, rmin)
    G0, = torch.autograd.grad(E0.sum(), pt0)
    q = np.random.default_rng(n).integers(0, len(c), n)
    E, pt, *_ = _gpu(eng, 2, c[q], p[q], eps, rmin)
    G, = torch.autograd.grad(E.sum(), pt)
    e0, g0 = E0.detach().cpu().numpy()[q], G0.cpu().numpy()[q].reshape(n, -1)
    e, g = E.detach().cpu().numpy(), G.cpu().numpy().reshape(n, -1)
    assert (np.abs(e - e0) <= 1e-10 * np.maximum(np.abs(e0), 1.0)).all()
    assert (np.linalg.norm(g - g0, axis=1) <= 1e-4 * np.linalg.norm(g0, axis=1)).all()


@pytest.mark.parametrize('n,per,m', [(0, 9, 3), (1, 9, 3), (64, 36, 64), (65, 60, 65), (2048, 3, 198), (2111, 9, 1)])
def test_backward_sums(case, n, per, m):
    """One chunk of poses (up to 64), several, more than the workspace has chunks
    for; FP64 weights, rounded to FP32: the scaled rows exactly, column sums to
    the rounding of their FP32 result and of FP64 additions.  (No poses: torch's
    empty tensors have no address, which is refused.)"""
    from pygcmc_amd import engine as _engine
    eng, L = case[1], adjoint._lib()
    g = torch.Generator(device='cpu').manual_seed(n)
    x, y = torch.randn(n, per, generator=g), torch.randn(n, m, generator=g) * 10
    w = torch.rand(n, generator=g, dtype=torch.float64)
    xd, yd, wd = x.cuda(), y.cuda(), w.cuda()
    gp, gc = torch.full((n, per), float('nan'), device='cuda'), torch.full((m,), float('nan'), device='cuda')
    rc = L.gcmc_engine_adjoint_backward64(eng._h, n, per, m, *(adjoint._ptr(t) for t in (xd, yd, wd, gp, gc)),
                                          adjoint.ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    if n == 0:
        assert rc < 0
        return
    _engine._check(rc)
    w32 = w.float()
    assert torch.equal(gp.cpu(), w32[:, None] * x)
    terms = w32.double()[:, None] * y.double()
    ref, size = terms.sum(0), terms.abs().sum(0)
    assert ((gc.cpu().double() - ref).abs() <= 2.0 ** -24 * ref.abs() * 1.001 + 1e-12 * size).all()


@pytest.mark.parametrize('few', [True, False])
def test_type_gradients_inside_sigma(case, few):
    """Type gradients of close contacts, where one pair outweighs the others,
    four waves per pose and one.  The terms inside sigma are rounded to FP32
    once (s^12 would carry six times the rounding of an FP32 s^2).  Roundings of
    2^-24 at most: table entry and its root 2, 1/sigma 2, constants and products
    6, a lane's and the wave's additions 16: 26 2^-24 of the largest derivative."""
    s, eng, eps, rmin, poses = case
    e64, r64 = eps.double().cpu().numpy(), rmin.double().cpu().numpy()
    ref, got = [], []
    c, p = poses[5]
    at = s['atoms']['position'][:int(s['res'][int(s['frag'][0]['startRes']) - 1]['atomStart'])].astype(np.float64)
    L = s['info'][0]['cryst'].astype(np.float64)
    for i in range(4):
        # moved so that the first atom lies 2.2 A from the nearest fixed one
        d = p[i][0].astype(np.float64) - at
        d -= np.rint(d / L) * L
        j = int(np.argmin((d ** 2).sum(1)))
        v = d[j] * (2.2 / np.linalg.norm(d[j]) - 1.0)
        q, x = (p[i] + v).astype(np.float32)[None], (c[i] + v).astype(np.float32)[None]
        ref.append(np.stack(O.adjoint(s, 5, x[0], q[0], e64, r64)[3:5]))
        n = 1 if few else 2048
        E, pt, e, r, _ = _gpu(eng, 5, np.repeat(x, n, 0), np.repeat(q, n, 0), eps, rmin)
        ge, gr = torch.autograd.grad(E.sum() / n, (e, r))
        got.append(np.stack([ge.cpu().numpy(), gr.cpu().numpy()]))
    for a, b in zip(got, ref):
        for k in range(2):
            assert np.linalg.norm(a[k] - b[k]) <= 26 * 2.0 ** -24 * np.linalg.norm(b[k]), k


def test_charge_derivatives_with_one_wave_per_pose():
    """dE/dq of a pose's types carries the same rounding whether four waves share
    the pose or one has it: in either form a lane adds the terms of at most 16
    environment atoms per fragment atom in FP32, the rest is added in FP64.  RMS
    error against 64 bits over 24 poses and all types, one wave's within 1.25 of
    four waves' (the sampling error of some 500 values of unlike size)."""
    from pygcmc_amd import engine as _engine
    s = systems.multi(nsteps=10, n_fixed=20000, box=86.0)
    eng = Engine()
    eng.add_system(s)
    eng.upload()
    eps, rmin = adjoint.type_parameters(s)
    e64, r64 = eps.double().cpu().numpy(), rmin.double().cpu().numpy()
    for spi in range(int(s['info'][0]['fragTypeNum'])):
        c, p = systems.moderate_poses(s, spi, 24, seed=41 + spi)
        ref = np.stack([O.adjoint(s, spi, c[i], p[i], e64, r64)[2] for i in range(24)])
        rms = []
        for n in (24, 2064):
            q = np.arange(n) % 24
            ct, pt = torch.tensor(c[q], device='cuda'), torch.tensor(p[q], device='cuda')
            E = torch.empty(n, dtype=torch.float64, device='cuda')
            dx = torch.empty(pt.shape, device='cuda')
            part = torch.empty((n, 3, len(e64)), device='cuda')
            _engine._check(adjoint._lib().gcmc_engine_adjoint(
                eng._h, 0, spi, n, *(adjoint._ptr(t) for t in (ct, pt, eps, rmin)), None,
                *(adjoint._ptr(t) for t in (E, dx, part)),
                adjoint.ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
            got = part[:, 0].cpu().numpy().astype(np.float64)
            assert np.abs(got - got[q]).max() <= 2.0 ** -23 * np.abs(got).max()   # copies agree
            rms.append(np.sqrt(((got[:24] - ref) ** 2).mean()))
        print(spi, rms)
        assert rms[1] <= 1.25 * rms[0], spi
    eng.close()
