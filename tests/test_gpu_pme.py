"""GPU PME reciprocal part against the FP64 Ewald sums (oracle/ewald.py).

Bars (order-4 B-splines, beta = 0.34 /A): reciprocal energy within 1e-3
relative at 1 A grid spacing and 6e-5 at 0.5 A (measured 5.7e-4 and 3.0e-5:
the h^4 convergence of cubic B-spline interpolation, checked as such);
potentials within 2e-3 of their spread; exact invariants: neutral pairs at
coincident points give zero, 1/2 sum q phi = E_rec.
"""

import numpy as np
import pytest
import torch

from oracle import ewald
from pygcmc_amd.pme import PME

pytestmark = pytest.mark.gpu


def _charges(n, L, seed):
    rng = np.random.default_rng(seed)
    xyz = rng.random((n, 3)) * L
    q = rng.normal(0, 0.5, n)
    q -= q.mean()
    return xyz, q


def _t(xyz, q=None):
    a = xyz if q is None else np.concatenate([xyz, q[:, None]], 1)
    return torch.tensor(a, dtype=torch.float32, device='cuda')


def test_pme_energy_against_ewald():
    L = [24.0, 21.0, 27.0]
    beta = 0.34
    xyz, q = _charges(200, L, 1)
    ref = ewald.recip_energy(xyz, q, L, beta, kmax=(14, 12, 16))
    rels = {}
    for spacing in (1.0, 0.5):
        grid = [int(round(l / spacing)) for l in L]
        p = PME(grid, L, beta)
        e = p.energy(_t(xyz, q))
        rels[spacing] = abs(e - ref) / abs(ref)
        print(f'spacing {spacing}: E_rec {e:.6f} ref {ref:.6f} rel {rels[spacing]:.2e}')
        p.close()
    assert rels[1.0] <= 1e-3 and rels[0.5] <= 6e-5
    # fourth-order convergence: halving the spacing cuts the error ~16x
    assert rels[1.0] / rels[0.5] >= 8.0


def test_pme_potential_against_ewald():
    L = [24.0, 21.0, 27.0]
    beta = 0.34
    xyz, q = _charges(150, L, 2)
    pts = np.random.default_rng(3).random((64, 3)) * L
    ref = ewald.recip_potential(xyz, q, L, beta, (14, 12, 16), pts)
    p = PME([24, 21, 27], L, beta)
    p.clear()
    p.spread(_t(xyz, q))
    E = p.solve()
    phi = p.gather(_t(pts)).cpu().numpy()
    err = np.abs(phi - ref).max() / (np.abs(ref).max() + 1e-9)
    print(f'potential: max err / max |phi| = {err:.2e}')
    assert err <= 2e-3
    # 1/2 sum_i q_i phi(x_i) = E_rec (same grid quantities)
    phi_s = p.gather(_t(xyz)).cpu().numpy().astype(np.float64)
    assert abs(0.5 * float((q * phi_s).sum()) - float(E.item())) <= 1e-4 * abs(float(E.item()))
    p.close()


def test_pme_neutral_coincident_pair_is_zero():
    L = [20.0, 20.0, 20.0]
    p = PME([20, 20, 20], L, 0.34)
    x = np.array([[3.3, 7.1, 11.9], [3.3, 7.1, 11.9]])
    e = p.energy(_t(x, np.array([1.0, -1.0])))
    assert abs(e) < 1e-6
    p.close()


def test_pme_slab_config_grid():
    """The 150 x 150 x 120 A box on a 1 A grid (2.7 M points), beta 0.34."""
    L = [150.0, 150.0, 120.0]
    xyz, q = _charges(100, L, 5)
    p = PME([150, 150, 120], L, 0.34)
    e = p.energy(_t(xyz, q))
    # terms beyond |k_i| = 0.4 L_i are below exp(-13.7) of the largest
    ref = ewald.recip_energy(xyz, q, L, 0.34, kmax=(60, 60, 48))
    assert abs(e - ref) <= 1e-3 * abs(ref)
    p.close()


def _spme64(xyzq, K, L, beta):
    """Potential of smooth PME at the charges themselves, in FP64."""
    K = np.array(K)
    u = np.mod(xyzq[:, :3].astype(np.float64) / L, 1.0) * K
    f = np.floor(u).astype(np.int64) % K
    t = u - np.floor(u)
    w = np.stack([t ** 3 / 6, (-3 * t ** 3 + 3 * t ** 2 + 3 * t + 1) / 6, (3 * t ** 3 - 6 * t ** 2 + 4) / 6,
                  (1 - t) ** 3 / 6])
    pts = [(tuple((f[:, d] - j[d]) % K[d] for d in range(3)), w[j[0], :, 0] * w[j[1], :, 1] * w[j[2], :, 2])
           for j in np.ndindex(4, 4, 4)]
    Q = np.zeros(K)
    for k, v in pts:
        np.add.at(Q, k, v * xyzq[:, 3])
    B, m = [], []
    for d in range(3):
        i = np.arange(K[d])
        z = sum(a * np.exp(2j * np.pi * i * n / K[d]) for n, a in enumerate((1 / 6, 2 / 3, 1 / 6)))
        B.append(1.0 / np.abs(z) ** 2)
        m.append(np.where(i <= K[d] // 2, i, i - K[d]) / L[d])
    m2 = m[0][:, None, None] ** 2 + m[1][None, :, None] ** 2 + m[2][None, None, :] ** 2
    m2[0, 0, 0] = 1.0
    G = 1388.431112 / (np.pi * np.prod(L)) * np.exp(-np.pi ** 2 * m2 / beta ** 2) / m2
    G *= B[0][:, None, None] * B[1][None, :, None] * B[2][None, None, :]
    G[0, 0, 0] = 0.0
    phi = np.fft.ifftn(G * np.fft.fftn(Q)).real * Q.size
    return sum(phi[k] * v for k, v in pts)


@pytest.mark.parametrize('K', [(4, 5, 4), (8, 8, 16), (9, 17, 18), (10, 25, 34), (31, 33, 50)])
@pytest.mark.parametrize('n', [16383, 16384, 40001])
def test_pme_spread_of_many_charges(K, n):
    """Charges sorted by grid tile (one call) give the same charge grid, bit
    for bit, as added a few at a time, and the FP64 potential: tiles cut by
    the box, last tiles of one or two points, an axis of one tile, more charges
    than are sorted at once, zero charges, positions outside the box.
    Tolerance: FP32 weights, transforms and sums of n charges, 2e-5 of the
    largest potential."""
    rng = np.random.default_rng(n + K[0])
    L = np.array([0.9 * k for k in K])
    a = np.concatenate([(rng.random((n, 3)) * 3.0 - 1.0) * L, rng.normal(0, 0.3, (n, 1))], 1).astype(np.float32)
    a[:, 3] -= a[:, 3].mean()
    a[::97, 3] = 0.0
    t = torch.tensor(a, device='cuda')
    out = []
    for step in (n, 5000):
        p = PME(K, L, 0.34)
        p.clear()
        for i in range(0, n, step):
            p.spread(t[i:i + step])
        e = p.solve()
        out.append((p.gather(t[:, :3].contiguous()).cpu().numpy(), float(e.item())))
        p.close()
    (phi, e), (phi1, e1) = out
    assert np.array_equal(phi.view(np.uint32), phi1.view(np.uint32)) and e == e1
    ref = _spme64(a, K, np.float32(L).astype(np.float64), float(np.float32(0.34)))
    assert np.abs(phi - ref).max() <= 2e-5 * np.abs(ref).max()


@pytest.mark.parametrize('K', [(4, 130, 260), (130, 129, 5), (9, 297, 50), (129, 145, 18), (64, 64, 64)])
@pytest.mark.parametrize('n', [24575, 24576, 'room', 'room+5'])
def test_pme_spread_by_tiles(K, n):
    """At and past the line from which charges are sorted by tile, on grids of 256
    tiles and more: axes of one tile, last tiles of one or two points, as many
    charges as are sorted at once (a quarter of the points) and a few more.  Bit
    for bit the grid of charges added a few at a time, and the FP64 potential:
    2e-5 of the largest for FP32 weights, transforms and sums, 2e-7 per point of
    the longest axis for FP32 scaled positions (two roundings of 2^-23)."""
    room = max(K[0] * K[1] * K[2] // 4, 24576)
    n = {'room': room, 'room+5': room + 5}.get(n, n)
    rng = np.random.default_rng(n + K[0])
    L = np.array([0.9 * k for k in K])
    a = np.concatenate([(rng.random((n, 3)) * 3.0 - 1.0) * L, rng.normal(0, 0.3, (n, 1))], 1).astype(np.float32)
    a[:, 3] -= a[:, 3].mean()
    a[::97, 3] = 0.0
    t = torch.tensor(a, device='cuda')
    out = []
    for step in (n, 5000):
        p = PME(K, L, 0.34)
        p.clear()
        for i in range(0, n, step):
            p.spread(t[i:i + step])
        e = p.solve()
        out.append((p.gather(t[:, :3].contiguous()).cpu().numpy(), float(e.item())))
        p.close()
    (phi, e), (phi1, e1) = out
    assert np.array_equal(phi.view(np.uint32), phi1.view(np.uint32)) and e == e1
    ref = _spme64(a, K, np.float32(L).astype(np.float64), float(np.float32(0.34)))
    assert np.abs(phi - ref).max() <= (2e-5 + 2e-7 * max(K)) * np.abs(ref).max()
