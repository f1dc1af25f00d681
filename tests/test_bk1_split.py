"""Production rates split over wavefronts (kinetix_amd/gen/emit_bk1_split.py) and the range-free
exponentials they use (kinetix_amd/csrc/kx_exp.h)."""
import os
import re
from decimal import Decimal, getcontext

import numpy as np
import pytest

from kinetix_amd import states
from kinetix_amd.gen import emit_bk1_split as SP
from kinetix_amd.gen import tables
from oracle import pyoracle as po

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
P_ATM = 101325.0


def load(mech):
    return tables.load(os.path.join(ROOT, 'kinetix_amd', 'mechs', mech))


@pytest.mark.parametrize('mech', ['gri30', 'NH3Konnov_edit', 'chempolimi_edit', 'synth40cov'])
def test_plan_covers_every_reaction_and_sum(mech):
    """Every reaction in one wavefront, every (wavefront, species) sum in one LDS slot of one
    round, slots inside the rows and never shared within a round, and the sums of all
    wavefronts added up give nu^T q."""
    info, t = load(mech)
    assert SP.pays(t, info)
    p = SP.plan(t, info)
    em = p['em']
    assert sorted(r for rs in p['rs'] for r in rs) == list(range(em.R))
    seen = {}
    for rnd in p['rounds']:
        assert len(set(rnd.values())) == len(rnd) and max(rnd.values()) < p['rows']
        for key in rnd:
            assert key not in seen
            seen[key] = True
    assert set(seen) == {(w, k) for w in range(p['waves']) for k in p['sums'][w]}
    assert sorted([*p['wrow'].values(), *p['rrow'].values(), *p['crow'].values()]) == \
        list(range(em.N + len(p['rrow']) + len(p['crow'])))
    q = np.random.default_rng(1).normal(size=em.R)
    wd = np.zeros(em.N)
    for w, rs in enumerate(p['rs']):
        part = {k: sum(em.net[r, k] * q[r] for r in rs) for k in p['sums'][w]}
        for k, v in part.items():
            wd[k] += v
    np.testing.assert_allclose(wd, em.net.T @ q, rtol=1e-12, atol=1e-12)
    assert not SP.pays(*reversed(load('LiDryer')))


@pytest.mark.parametrize('mech,waves,occupancy', [('gri30', 8, 4), ('EtOHKonnov', 12, 3), ('synth160', 8, 2)])
def test_shapes(mech, waves, occupancy):
    """The layout by size: rows within the LDS, a species' sums of all wavefronts in one round,
    and every third body's concentration from its own row or from w and rg rows."""
    info, t = load(mech)
    p, occ, segment = SP.pays(t, info)
    em = p['em']
    assert (p['waves'], occ) == (waves, occupancy) and segment in (3, SP.SEGMENT)
    assert p['tight'] == (occupancy < 4)
    assert SP.lds_bytes(em.N, p['rows'], waves, p['tight']) <= SP.LDS_MAX // (2 if occupancy == 4 else 1)
    for k in range(em.N):
        assert len({i for i, rnd in enumerate(p['rounds']) for w, j in rnd if j == k}) <= 1
    for r in range(em.R):
        if em.kind[r] not in (SP.M.ELEMENTARY, SP.M.PLOG):
            third = np.flatnonzero(em.t['eff'][r] != 1.0) if em.has_eff[r] else \
                [k for k in (int(em.t['collider'][r]),) if k >= 0]
            assert all(k in p['crow'] or k in p['rrow'] for k in third)


def padded(t, N):
    """A mechanism's tables with inert species appended up to N."""
    n, R = int(t['n_species']), int(t['n_reactions'])
    out = dict(t, n_species=N)
    for k in ('nu_f', 'nu_r', 'eff'):
        a = np.asarray(t[k]).reshape(R, n)
        out[k] = np.concatenate([a, np.full((R, N - n), 1 if k == 'eff' else 0, a.dtype)], axis=1)
    for k in ('W', 'rcpW', 'T_mid', 'g_lo', 'g_hi', 'h_lo', 'h_hi'):
        a = np.asarray(t[k])
        out[k] = np.concatenate([a, np.repeat(a[-1:], N - n, axis=0)])
    return out


@pytest.mark.parametrize('waves', [8, 12])
@pytest.mark.parametrize('N', [290, 308, 315, 319])
def test_tight_rows_hold_the_partial_sums(N, waves):
    """Many species, few of them reactants: the tight layout's wavefront sums and ln T (waves + 1
    rows from row N on) lie within the rows, or the plan does not fit the LDS."""
    info, t = load('LiDryer')
    p = SP.plan(padded(t, N), info, waves)
    assert p['tight'] and p['rows'] >= N + waves + 1
    if N + waves + 1 > SP.LDS_MAX // (8 * SP.ROW):
        assert SP.lds_bytes(N, p['rows'], waves, True) > SP.LDS_MAX


@pytest.mark.parametrize('reactants,products', [({0: 5}, {1: 3}), ({0: 1}, {k: 1 for k in range(1, 11)})])
def test_global_reactions_beside_plog(reactants, products):
    """A mechanism with PLOG reactions takes a reaction of more molecules or species than the loop
    forms' descriptors hold (4 molecules a side, 8 species): straight-line code has no limit."""
    info, t = load('NH3Konnov_edit')
    assert np.any(t['kind'] == SP.M.PLOG)
    t = {k: np.array(v) if isinstance(v, np.ndarray) else v for k, v in t.items()}
    r = int(np.flatnonzero(t['kind'] == SP.M.ELEMENTARY)[5])
    t['reversible'][r] = 0
    for key, nu in (('nu_f', reactants), ('nu_r', products)):
        t[key][r] = 0
        for k, v in nu.items():
            t[key][r, k] = v
    src = SP.emit(t, info, 'fp64', SP.pays(t, info))
    line = next(ln for ln in src.split(f'{{ // {r + 1}: ')[1].split('\n') if 'double F' in ln)
    assert line.count('rg0') == reactants[0]


@pytest.mark.parametrize('A', [0.0, -1e3])
def test_rate_coefficients_without_a_logarithm_are_refused(A):
    """A <= 0 is no Arrhenius coefficient, with or without an exponential beside it."""
    info, t = load('gri30')
    for beta, Ta in ((0.0, 0.0), (1.0, 0.0), (0.5, 100.0)):
        c = dict(t, A=t['A'].copy(), beta=t['beta'].copy(), Ta=t['Ta'].copy())
        r = int(np.flatnonzero(t['kind'] == SP.M.ELEMENTARY)[0])
        c['A'][r], c['beta'][r], c['Ta'][r] = A, beta, Ta
        for variant in ('fp64', 'mixed_valu'):
            em = SP.E._RateEmitter(c, info)
            em.arrh32 = variant == 'mixed_valu'
            with pytest.raises(ValueError):
                em.rate_const_p(r)


def test_troe_terms_switched_off_have_int_exponents():
    """Parameters that switch a Troe term off (T3 = 1e-30, T2 = 1e30 in these mechanisms): the
    exponents handed to kx_exp2, whose power of two is an int, stay in its range from 1 to
    20,000 K and far below -1,075, where 2^y is 0."""
    off = 0
    for mech in ('LiDryer', 'NH3Konnov_edit', 'chempolimi_edit'):
        info, t = load(mech)
        em = SP.E._RateEmitter(t, info)
        _, sidx = em.efficiency_sets()
        for r in np.flatnonzero(t['kind'] == SP.M.TROE):
            S = SP.E._Src()
            em.emit_reaction_p(S, int(r), sidx)
            line = next(ln for ln in S.lines if 'l2F = kx_log2' in ln)
            for c, at in re.findall(r'kx_exp2\(([-0-9.e+]+) \* (T|rcpT)\)', line):
                y = [float(c) * (T if at == 'T' else 1.0 / T) for T in (1.0, 300.0, 20000.0)]
                assert max(abs(v) for v in y) < 2 ** 31
                off += max(y) < -2000
            rT3, rT1, T2 = t['troe'][r][1:]
            assert len(re.findall('kx_exp2', line)) == (3 if T2 >= 0 else 2)
    assert off >= 10


@pytest.mark.parametrize('mech', ['gri30', 'NH3Konnov_edit', 'EtOHKonnov'])
def test_order_reads_fewer_rows(mech):
    """A wavefront's searched order keeps its reactions, is the same each time, and reads no more
    LDS rows (distinct rows of every segment, hot rows once) than the greedy order."""
    info, t = load(mech)
    p, _, segment = SP.pays(t, info)
    em = p['em']

    def reads(o, hot):
        rows = [set().union(*[SP.rows_of(em, r) for r in o[i:i + segment]]) for i in range(0, len(o), segment)]
        return len(hot) + sum(len(x - hot) for x in rows)
    for rs in p['rs']:
        plain, none = SP.order(em, rs, segment, None)
        o, hot = SP.order(em, rs, segment)
        assert sorted(plain) == sorted(o) == sorted(rs) and not none
        assert len(hot) <= SP.HOT_ROWS and hot <= set().union(*[SP.rows_of(em, r) for r in rs])
        assert (o, hot) == SP.order(em, rs, segment)
        assert reads(o, hot) <= reads(plain, none)


def _poly(body):
    """Coefficients of a Horner chain, lowest first, from the C source."""
    c = re.findall(r'(?:double p =|fma\(p, \w,) ([-0-9.e]+)\)?;', body)
    return [Decimal(v) for v in reversed(c)]


def test_exponential_polynomials():
    """The polynomials of kx_exp.h against exp2, exp and log2 in 50 digits: relative error below
    2.1e-17 (a fifth of FP64 rounding) over the reduced ranges, and ln 2's two parts exact."""
    getcontext().prec = 50
    src = open(os.path.join(ROOT, 'kinetix_amd', 'csrc', 'kx_exp.h')).read()
    body = {n: src.split(f'double {n}(double')[1].split('\n}\n')[0] for n in ('kx_exp2', 'kx_exp', 'kx_log2')}
    ln2 = Decimal(2).ln()
    ev = lambda p, x: sum((c * x ** k for k, c in enumerate(p) if k), p[0])
    grid = [Decimal(i) / 200 for i in range(-100, 101) if i]
    p = [Decimal(float(c)) for c in _poly(body['kx_exp2'])]
    assert len(p) == 12
    assert max(abs(ev(p, x) / (x * ln2).exp() - 1) for x in grid) < Decimal('2.1e-17')
    p = [Decimal(float(c)) for c in _poly(body['kx_exp'])]
    assert len(p) == 12
    assert max(abs(ev(p, x * ln2) / (x * ln2).exp() - 1) for x in grid) < Decimal('2.1e-17')
    hi, lo = Decimal(0.6931471228599548), Decimal(5.7699990475432854e-08)
    assert '0.6931471228599548' in body['kx_exp'] and '5.7699990475432854e-08' in body['kx_exp']
    assert abs(hi + lo - ln2) <= Decimal(2) ** -78            # half a unit in the last place of lo
    assert int(np.frexp(0.6931471228599548)[0] * 2 ** 24) == np.frexp(0.6931471228599548)[0] * 2 ** 24
    p = [Decimal(float(c)) for c in _poly(body['kx_log2'])]
    assert len(p) == 8
    for i in range(1, 100):
        m = (Decimal('0.5').sqrt() * (100 - i) + Decimal(2).sqrt() * i) / 100
        if m == 1:
            continue
        s = (m - 1) / (m + 1)
        assert abs(s * ev(p, s * s) / (m.ln() / ln2) - 1) < Decimal('2.1e-17')


@pytest.mark.gpu
@pytest.mark.parametrize('mech,n,p_atm', [('gri30', 1, 1.0), ('gri30', 63, 1.0), ('gri30', 1000, 20.0),
                                          ('NH3Konnov_edit', 65, 0.05), ('NH3Konnov_edit', 257, 3.0),
                                          ('chempolimi_edit', 64, 2000.0), ('synth40cov', 129, 1.0),
                                          ('LiDryer', 300, 5.0), ('EtOHKonnov', 1, 1.0),
                                          ('EtOHKonnov', 129, 20.0), ('synth160', 191, 0.3)])
def test_split_rates_at_group_edges(mech, n, p_atm):
    """FP64 and mixed rates at state counts around the 64-state groups on a strided view, cold
    and hot (300-3000 K, both NASA-7 pieces), against the oracle; nothing outside the view."""
    import torch
    from kinetix_amd.api import Kinetix
    info, t = load(mech)
    N, lo = int(t['n_species']), 3
    ld = n + 11
    s, _ = states.sample_any(ld, info['species'], t['W'], T_range=(300.0, 3000.0), seed=41 + n)
    kx = Kinetix(mech, device=0)
    got = {}
    try:
        kx.build(P_ATM, 1.0, states.reference_mass_fractions(info['species'], t['W']))
        ds = torch.from_numpy(s).cuda().reshape(-1)[lo:]
        for mixed in (False, True):
            r = torch.full((N + 1, ld), np.nan, dtype=torch.float64, device='cuda')
            kx.productionRates(n, ld, ld, p_atm, ds, r.reshape(-1)[lo:], mixed=mixed)
            torch.cuda.synchronize()
            got[mixed] = r.cpu().numpy()
    finally:
        kx.close()
    orc = po.Oracle(t)
    sub = np.ascontiguousarray(s[:, lo:lo + n])
    ref, scale = orc.production_rates(sub, p_atm * P_ATM, scale=True)
    # mixed: FP32 exponents up to 300 at 300 K, 300 ln 2 / 2^23 = 2.5e-5, and FP32 falloff
    for mixed, tol in ((False, 1e-12), (True, 4e-5)):
        a = got[mixed]
        assert np.all(np.isnan(a[:, :lo])) and np.all(np.isnan(a[:, lo + n:]))
        # against the magnitude of the terms each rate is the sum of
        assert np.all(np.isfinite(a[:, lo:lo + n]))
        err = np.abs(a[:, lo:lo + n] - ref) / np.maximum(np.maximum(np.abs(ref), scale), 1e-300)
        assert err.max() < tol, (mixed, float(err.max()))
