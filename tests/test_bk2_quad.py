"""The four-lanes-per-state transport routine (kinetix_amd/csrc/kx_bk2_quad.h): its table and
index arithmetic emulated on the CPU against the oracle, and the kernels on the GPU at the
edges of their 16-state groups."""
import os

import numpy as np
import pytest

from kinetix_amd import states
from kinetix_amd.gen import emit_bk2_quad as Q
from kinetix_amd.gen import tables
from oracle import pyoracle as po

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MECHS = ['gri30', 'NH3Konnov_edit', 'chempolimi_edit', 'LiDryer', 'synth40cov']


def load(mech):
    return tables.load(os.path.join(ROOT, 'kinetix_amd', 'mechs', mech))


def _mfma(a, b, c):
    """v_mfma_f64_16x16x4_f64: A[i][k] = a[i + 16 k], B[k][j] = b[j + 16 k],
    D[4 r + l // 16][l % 16] -> c[l][r] (the layout kx_selftest_mfma_f64_layout checks)."""
    D = a.reshape(4, 16).T @ b.reshape(4, 16)
    d = c.copy()
    for l in range(64):
        for r in range(4):
            d[l, r] += D[4 * r + l // 16, l % 16]
    return d


def quad_numpy(t, s, p):
    """16 states as the wavefront computes them, lane arrays of 64; returns mu, lambda, rhoD, Dkm."""
    N = int(t['n_species'])
    nb = Q.slots(N)
    sg, blk = (nb + 3) // 4, nb * (nb + 1) // 2
    tab = Q.table(t)
    kr = Q.rank_groups(t)
    rb = (kr + 3) // 4
    o = np.cumsum([80 * blk, 64 * nb * rb, 64 * sg * kr, 64 * sg, 16 * sg, 64 * sg, 16 * sg,
                   4 * nb, 4 * nb, 4 * nb])
    wilT, wil, vA, vC, lA, lC, rW, Wt, sW = (tab[a:b] for a, b in zip(o[:-1], o[1:]))
    lane = np.arange(64)
    st, g = lane % 16, lane // 16
    T = s[0][st]
    x = np.zeros((nb, 64))
    for m in range(nb):
        k = 4 * m + g
        x[m] = np.where(k < N, np.maximum(s[1 + np.minimum(k, N - 1), st], 0.0), 0.0) * rW[4 * m + g]
    sum4 = lambda v: np.tile(v.reshape(4, 16).sum(0), 4)
    bc = lambda v: v.reshape(4, 16)[:, st]                    # [c][lane]: value of lane group c
    rs = lambda q: np.stack(q).reshape(4, 4, 16).sum(1).reshape(64)   # p[c] summed over groups, to group c
    Mbar = 1.0 / sum4(x.sum(0))
    x *= Mbar
    tt = np.log(T) - Q.center(t)
    B = tt ** (g + 1)
    acc = lambda C, i: C[16 * i:16 * i + 16].reshape(4, 4)[g]
    S = np.zeros((nb, 64))
    for m in range(nb):
        xk, q = bc(x[m]), np.zeros((4, 64))
        for j in range(m + 1):
            row = tab[40 * m * (m + 1):]
            d = _mfma(row[64 * j:64 * j + 64], B, acc(row[64 * (m + 1):], j))
            r = (d if int(t['rcp_diff']) else 1.0 / d).T
            if j < m:
                S[j] += (xk * r).sum(0)
                q += x[j] * r
            else:
                S[m] += (xk * np.where(np.arange(4)[:, None] == g, 0.0, r)).sum(0)
        S[m] += rs(q)
    pl = p[st]
    rho = pl / float(t['R']) / T * Mbar
    D = np.stack([T ** 1.5 * (Mbar - Wt[4 * m + g] * x[m]) / (pl * Mbar * np.where(4 * m + g < N, S[m], 1.0))
                  for m in range(nb)])
    s1, s2, U, A = np.zeros(64), np.zeros(64), np.zeros((nb, 64)), np.zeros((nb, 64))
    for h in range(sg):
        l = _mfma(lA[64 * h:64 * h + 64], B, acc(lC, h))
        u = _mfma(vA[64 * h:64 * h + 64], B, acc(vC, h))
        for c in range(4):
            m = 4 * h + c
            if m < nb:
                s1 += x[m] * l[:, c]
                s2 += x[m] / l[:, c]
                U[m], A[m] = u[:, c], x[m] * sW[4 * m + g] / u[:, c] ** 2
    vis, z = np.zeros(64), np.zeros((3, rb, 64, 4))
    for v in range(3):
        for h in range(rb):
            for m in range(nb):
                z[v, h] = _mfma(wilT[64 * (rb * m + h):][:64], A[m] * U[m] ** v, z[v, h])
    for h in range(sg):
        y = np.zeros((3, 64, 4))
        for v in range(3):
            for q in range(kr):
                y[v] = _mfma(wil[64 * (kr * h + q):][:64], z[v, q // 4, :, q % 4], y[v])
        for c in range(4):
            m = 4 * h + c
            if m < nb:
                S = y[2, :, c] + U[m] * (2 * y[1, :, c] + U[m] * y[0, :, c])
                vis += A[m] * U[m] ** 4 / np.where(4 * m + g < N, S, 1.0)
    mu, lam = np.sqrt(T) * sum4(vis), np.sqrt(T) * 0.5 * (sum4(s1) + 1.0 / sum4(s2))
    rows = lambda v: np.concatenate([v[m].reshape(4, 16) for m in range(nb)])[:N]
    return lam[:16], mu[:16], rows(D * rho), rows(D)


@pytest.mark.parametrize('mech', MECHS + ['EtOHKonnov', 'synth160', 'synth22heavy'])
def test_quad_routine_vs_oracle(mech):
    info, t = load(mech)
    s, p = states.sample_any(16, info['species'], t['W'], T_range=(300.0, 2500.0), seed=31,
                             p_range_atm=(0.5, 40.0))
    ref = po.Oracle(t).transport(s, 1.0, 1.0, p_state=p)
    # the oracle sums the fits in powers of ln T: up to 2e-15 times their condition number
    # (1e5 for helium's conductivity); the table's own expansion about t0 does not cancel
    lt = np.log(s[0])
    P = np.stack([lt ** i for i in range(5)])
    kappa = 1.0
    for key in ('cond', 'visc', 'diff'):
        c = np.asarray(t[key]).reshape(-1, 5)
        c = c[np.any(c != 0, axis=1)]
        kappa = max(kappa, float(((np.abs(c) @ np.abs(P)) / np.abs(c @ P)).max()))
    for got, want in zip(quad_numpy(t, s, p), ref):
        assert np.max(np.abs(got / want - 1)) < 1e-12 + 2e-15 * kappa


@pytest.mark.parametrize('mech,rank', [('gri30', 13), ('synth160', 13), ('synth22heavy', 21)])
def test_wilke_factor_ranks(mech, rank):
    """The factor reproduces its matrix to rounding at any rank; 22 molar masses spread over a factor of
    300 in geometric steps have rank 21 and need a second block of 16 ranks."""
    _, t = load(mech)
    W = np.asarray(t['W'])
    L = Q.wilke_factor(W)
    assert L.shape[1] == rank
    M = (8 * (W[:, None] + W)) ** -0.5
    assert np.max(np.abs(L @ L.T / M - 1)) < 2e-15
    assert np.max(np.abs(L) @ np.abs(L).T / M) < 2.0


@pytest.mark.gpu
@pytest.mark.parametrize('mech,n', [('gri30', 1), ('gri30', 15), ('gri30', 2049), ('gri30', 33000),
                                    ('chempolimi_edit', 17), ('synth40cov', 4097),
                                    ('EtOHKonnov', 1), ('EtOHKonnov', 2065), ('synth160', 33000),
                                    ('synth22heavy', 17), ('synth22heavy', 4097)])
def test_quad_kernels_at_group_edges(mech, n):
    """Scalar, per-state-pressure and (straight-line mechanisms) MFMA entry points, the table
    resident in LDS and streamed (129 and 160 species), at state counts that end inside a 16-state group, fill every wavefront of the grid (256 x 8 x 16 states on a 256-CU GPU) and
    run past it, on a strided view: against the oracle, nothing written outside the view, and
    the same bits whatever the group a state lands in."""
    import torch
    from conftest import cond_err
    from kinetix_amd.api import Kinetix
    info, t = load(mech)
    N, lo = int(t['n_species']), 5
    ld = n + 13
    s, p = states.sample_any(ld, info['species'], t['W'], T_range=(300.0, 2500.0), seed=33 + n,
                             p_range_atm=(0.5, 40.0))
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    z = lambda *sh: torch.full(sh, np.nan, dtype=torch.float64, device='cuda')
    kx = Kinetix(mech, device=0)
    try:
        kx.build(101325.0, 1.0, states.reference_mass_fractions(info['species'], t['W']))
        ds, dp = d(s).reshape(-1)[lo:], d(p)[lo:]
        out = {}
        for form in ('plain', 'mfma', 'pstate') if N <= 96 else ('plain', 'pstate'):
            v, c, r, D = z(n), z(n), z(N, ld), z(N, ld)
            R, DD = r.reshape(-1)[lo:], D.reshape(-1)[lo:]
            if form == 'pstate':
                kx.mixtureAvgTransportPropsPstate(n, ld, ld, dp, ds, v, c, R, DD)
            else:
                kx.mixtureAvgTransportProps(n, ld, ld, 1.0, ds, v, c, R, mfma=form == 'mfma')
            torch.cuda.synchronize()
            out[form] = [a.cpu().numpy() for a in (c, v, r, D)]
        # a view shifted by one state: other groups, the same arithmetic per state
        if n > 1:
            v, c, r = z(n - 1), z(n - 1), z(N, ld)
            kx.mixtureAvgTransportProps(n - 1, ld, ld, 1.0, ds[1:], v, c, r.reshape(-1)[lo + 1:])
            torch.cuda.synchronize()
            assert np.array_equal(v.cpu().numpy(), out['plain'][1][1:])
            assert np.array_equal(r.cpu().numpy()[:, lo + 1:lo + n], out['plain'][2][:, lo + 1:lo + n])
    finally:
        kx.close()
    i = np.unique(np.concatenate([np.arange(min(n, 64)), np.arange(max(0, n - 64), n)])) + lo
    ref = po.Oracle(t).transport(np.ascontiguousarray(s[:, i]), 1.0, 1.0, p_state=p[i])
    for form, (c, v, r, D) in out.items():
        # helium's conductivity fit (condition number 1e5) bounds the oracle's own rounding
        tol = 1e-12 if mech == 'gri30' else 5e-12
        for got, want in zip((c[i - lo], v[i - lo], r[:, i]), ref):
            assert cond_err(got, want) < tol
        if form == 'pstate':
            assert cond_err(D[:, i], ref[3]) < tol
        for a in (r, D) if form == 'pstate' else (r,):
            assert np.all(np.isfinite(a[:, lo:lo + n]))
            assert np.all(np.isnan(a[:, :lo])) and np.all(np.isnan(a[:, lo + n:]))
    if 'mfma' in out:
        assert all(np.array_equal(a, b, equal_nan=True) for a, b in zip(out['plain'][:3], out['mfma'][:3]))
    assert all(np.array_equal(a, b) for a, b in zip(out['plain'][:2], out['pstate'][:2]))
