"""Production rates (BK1) with the reactions split over the wavefronts of a workgroup: kx_bk1_fp64
and kx_bk1_mixed_valu as straight-line code (benchmark/okl/productionRates.okl:10-62,
kinetix/core/reaction_rates.py:616-1333).

One lane still works on one state, but a workgroup's 8 or 12 wavefronts share the same 64 states:

  species    wavefront v takes the species k = v, v + waves, ...: Y, the Gibbs term g_k from the
             LDS NASA-7 table, e = exp(g_k), and puts w_k = C_k e and rg_k = 1 / e into LDS rows of 64
             states (512 B: every access is conflict-free);
  reactions  each wavefront runs its own part of the reactions as straight-line code (product
             form: q = k_f prod rg_reactants (prod w_reactants - C0^-dnu prod w_products)),
             reading w and rg from LDS where they are used and adding nu q to its own sums;
  sums       the wavefronts' sums meet in LDS rows (over the dead w and rg rows) and the
             species' owners add them in a fixed order, store W_k omega_k and add up the heat
             release.

Why: one wavefront that runs all of a state's reactions keeps three FP64 values per species alive
(474 registers for GRI-3.0: one wave per SIMD, which issues at most every fifth cycle, or, at two
waves, spills that double the HBM traffic). In LDS the values are shared, a wavefront needs
under 128 registers, and four waves per SIMD hide each other's latencies; a small call's latency
falls with the length of one wavefront's program.

Measured (before: one wavefront per 64 states, product form): GRI-3.0, 1,048,576 states FP64 762
-> 610 us, mixed 517 -> 425, 1,000 states FP64 41 -> 13.0 us; NH3Konnov_edit 2,510 -> 518 and
2,236 -> 378 us. Bound: FP64 issue and its power (75 % of the issue slots at 2.06 GHz). 4
wavefronts of 256 registers: 625 / 478 us, 15.4 us; 16: 949 / 774; two groups of 64 states per
workgroup in step: 715 / 566; a loop over groups instead of one per workgroup: 826 / 618 (the
compiler hoists the constants and spills).

Large mechanisms (shape) have one workgroup per CU; where the rows fill the LDS (plan's tight),
partial sums share them, the NASA-7 table stays in global memory and a third body's C_k is w_k
rg_k. Before, a loop over reaction descriptors with a state's species shared by 32 lanes (LDS
gathers and atomics, 160+ instructions a reaction; here 26 to 56, as constants are in the code and
equal exponentials are shared): 129 species / 1,231 reactions, 100,003 states FP64 1,732 -> 246
us, mixed 1,310 -> 211, 1,000 states 1,253 -> 30; 160 / 1,000, 524,288 states 5,340 -> 1,825,
mixed 4,164 -> 1,469, 1,000 states 1,298 -> 50. Of a group's 133,000 cycles at 160 / 1,000,
loading Y takes 13,000 (nothing beside it hides that), the species 20,000, the reactions
74,000 (61,000 of FP64 issue), the sums 11,000 (40,000 while each round took all sums of two or
three wavefronts: one reloaded its spilled sums while the others waited), the rest the end.

The reactions are dealt to the wavefronts by modelled cost with as few (wavefront, species) sums
as possible (assign), and the values read from LDS are cached for a segment of reactions.
"""
from __future__ import annotations

import math
import random

import numpy as np

from . import emit_hip as E
from . import emit_rolled as RL
from . import mechanism as M

WAVES = 8                # wavefronts that share 64 states' reactions
SEGMENT = 6              # reactions between points where values read from LDS are dropped
ROW = 64                 # states per workgroup
HOT_ROWS = 2             # rows a wavefront keeps in registers
LDS_MAX = 160 * 1024
MAX_SUMS = 100           # sums of a wavefront that stay in registers (two each, of 256)


def reaction_cost(em, r):
    """Issue cycles of one reaction (FP64), roughly: exponentials dominate."""
    t = em.t
    kind = em.kind[r]
    c = 30 + 8 * int(em.nu_f[r].sum() + em.nu_r[r].sum()) + 5 * int((em.net[r] != 0).sum())
    if kind == M.PLOG:
        return c + 300
    if em.arrh_key(t['beta'][r], t['Ta'][r]) is not None:
        c += 95
    if kind in (M.LINDEMANN, M.TROE, M.SRI):
        c += 140
    if kind in (M.TROE, M.SRI):
        c += 640
    return c


def assign(em, waves=WAVES, seed=7):
    """Wavefront of every reaction: greedy by cost, then a seeded local search over moves and
    swaps, minimising the largest load (in cycles) plus 12 cycles per (wavefront, species) sum
    and 40 per (wavefront, third-body set)."""
    R = em.R
    cost = np.array([reaction_cost(em, r) for r in range(R)], dtype=float)
    net = [np.flatnonzero(em.net[r]).tolist() for r in range(R)]

    def third(r):
        if em.kind[r] in (M.ELEMENTARY, M.PLOG) or not em.has_eff[r]:
            return None
        return tuple(em.t['eff'][r])
    sets = [third(r) for r in range(R)]
    load = np.zeros(waves)
    cnt = [dict() for _ in range(waves)]
    scnt = [dict() for _ in range(waves)]
    where = [0] * R

    def put(r, w, s):
        load[w] += s * cost[r]
        for k in net[r]:
            cnt[w][k] = cnt[w].get(k, 0) + s
            if not cnt[w][k]:
                del cnt[w][k]
        if sets[r] is not None:
            scnt[w][sets[r]] = scnt[w].get(sets[r], 0) + s
            if not scnt[w][sets[r]]:
                del scnt[w][sets[r]]
    target = cost.sum() / waves
    for r in sorted(range(R), key=lambda r: (-cost[r], r)):
        key = [(load[w] + cost[r] > 1.02 * target,
                12 * sum(k not in cnt[w] for k in net[r]) + 40 * (sets[r] is not None and sets[r] not in scnt[w])
                + 60 * load[w] / target, w) for w in range(waves)]
        w = min(key)[2]
        where[r] = w
        put(r, w, 1)

    def score():
        per = [load[w] + 12 * len(cnt[w]) + 40 * len(scnt[w]) for w in range(waves)]
        over = sum(max(0, len(c) - MAX_SUMS) for c in cnt)
        return waves * max(per) + sum(12 * len(c) for c in cnt) * 3 + 2000 * over
    rng = random.Random(seed)
    cur = score()
    # with sums beyond MAX_SUMS the search starts as an annealing (the descent gets stuck there)
    hot = 300.0 if max(len(c) for c in cnt) > MAX_SUMS else 0.0
    iters = 500 * R if hot else max(40000, 120 * R)
    for it in range(iters):
        r = rng.randrange(R)
        a = where[r]
        if rng.random() < 0.5:
            b, s = rng.randrange(waves), None
            if b == a:
                continue
        else:
            s = rng.randrange(R)
            b = where[s]
            if b == a:
                continue
        put(r, a, -1); put(r, b, 1)
        if s is not None:
            put(s, b, -1); put(s, a, 1)
        new = score()
        if new <= cur or (hot and rng.random() < math.exp((cur - new) / (hot * (1.0 - it / iters)))):
            cur = new
            where[r] = b
            if s is not None:
                where[s] = a
        else:
            put(r, b, -1); put(r, a, 1)
            if s is not None:
                put(s, a, -1); put(s, b, 1)
    return where


def rows_of(em, r):
    """The LDS rows a reaction reads: w of its reactants and (reversible) products, rg of its
    reactants."""
    ks = np.flatnonzero((em.nu_f[r] > 0) | (em.rev[r] & (em.nu_r[r] > 0)))
    return {('w', int(k)) for k in ks} | {('rg', int(k)) for k in np.flatnonzero(em.nu_f[r])}


def order(em, rs, segment=SEGMENT, hot_rows=HOT_ROWS, seed=7):
    """Order of one wavefront's reactions and its hot rows, the rows that most segments read,
    which stay in registers: greedy (next the reaction sharing most species with the last few),
    then a seeded search over swaps between segments for the fewest rows read. hot_rows None:
    greedy only (registers are short: 160 species 1,835 us, with the search 1,893, as the longer
    reuse spills more sums). 53 species: 975 rows read per group greedy, 859 searched, 779 with two
    hot; 4,194,304 states mixed, which is near the LDS rate, 1,754 us -> 1,711 -> 1,690, FP64 2,454 ->
    2,399 -> 2,393 (four hot, which spill, 1,801 and 2,415; segments of 8 or 10 no faster)."""
    used = {r: set(np.flatnonzero((em.nu_f[r] > 0) | (em.rev[r] & (em.nu_r[r] > 0))).tolist()) for r in rs}
    left, out, recent = sorted(rs), [], []
    while left:
        near = set().union(*recent[-segment:]) if recent else set()
        r = max(left, key=lambda r: (len(used[r] & near), -r))
        left.remove(r)
        out.append(r)
        recent.append(used[r])
    if hot_rows is None:
        return out, frozenset()
    rows = {r: rows_of(em, r) for r in rs}
    segs = [out[i:i + segment] for i in range(0, len(out), segment)]
    read = lambda s, hot: len(set().union(*[rows[r] for r in s]) - hot)

    def search(hot, iters=6000):
        rng = random.Random(seed)
        c = [read(s, hot) for s in segs]
        for _ in range(iters if len(segs) > 1 else 0):
            a, b = rng.sample(range(len(segs)), 2)
            i, j = rng.randrange(len(segs[a])), rng.randrange(len(segs[b]))
            A, B = list(segs[a]), list(segs[b])
            A[i], B[j] = B[j], A[i]
            ca, cb = read(A, hot), read(B, hot)
            if ca + cb <= c[a] + c[b]:
                segs[a], segs[b], c[a], c[b] = A, B, ca, cb
    search(frozenset())
    n = {}
    for s in segs:
        for x in set().union(*[rows[r] for r in s]):
            n[x] = n.get(x, 0) + 1
    hot = frozenset(sorted(n, key=lambda x: (-n[x], x))[:hot_rows])
    search(hot)
    return [r for s in segs for r in s], hot


def plan(t, info, waves=WAVES):
    """Everything the kernel text is written from: per wavefront the ordered reactions, its sums
    (species), and the rounds in which sums go through LDS rows (slot of every (wave, species))."""
    em = E._RateEmitter(t, info)
    N = em.N
    where = assign(em, waves)
    parts = [[r for r in range(em.R) if where[r] == w] for w in range(waves)]
    sums = [sorted({int(k) for r in parts[w] for k in np.flatnonzero(em.net[r])}) for w in range(waves)]
    react = sorted({int(k) for r in range(em.R) for k in np.flatnonzero(em.nu_f[r])})
    third = sorted({int(k) for r in range(em.R) if em.kind[r] not in (M.ELEMENTARY, M.PLOG)
                    for k in ([int(j) for j in np.flatnonzero(em.t['eff'][r] != 1.0)] if em.has_eff[r]
                              else [int(em.t['collider'][r])] if em.t['collider'][r] >= 0 else [])})
    # tight: no room for everything; the NASA-7 table stays in global memory, the wavefronts'
    # partial sums share the rows, and C_k of a species with an rg row is w_k rg_k
    tight = lds_bytes(N, N + len(react) + len(third), waves, False) > LDS_MAX
    if tight:
        third = [k for k in third if k not in react]
    wrow = {k: i for i, k in enumerate(range(N))}
    rrow = {k: N + i for i, k in enumerate(react)}
    crow = {k: N + len(react) + i for i, k in enumerate(third)}
    rows = max(N + len(react) + len(third), waves + 1)
    if tight:
        # emit's `part` (waves + 1 rows) starts where the rg rows do; one workgroup per CU: all
        # of the LDS, for fewer rounds of the sums
        rows = max(rows, N + waves + 1, LDS_MAX // (8 * ROW))
    # a round takes all wavefronts' sums of some species: every wavefront writes in every round
    rounds, cur, free = [], {}, rows
    for k in range(N):
        ws = [w for w in range(waves) if k in sums[w]]
        if len(ws) > free:
            rounds.append(cur)
            cur, free = {}, rows
        for w in ws:
            cur[(w, k)] = rows - free
            free -= 1
    rounds.append(cur)
    return dict(em=em, rs=parts, sums=sums, wrow=wrow, rrow=rrow, crow=crow, rows=rows, rounds=rounds,
                waves=waves, where=where, tight=tight)


def lds_bytes(N, rows, waves, tight):
    return 8 * ROW * rows if tight else 8 * (ROW * (rows + waves + 1) + 2 * N * 14)


def shape(t, info):
    """(plan, wavefronts per SIMD, reactions per segment) of a mechanism, or None when it does
    not fit.

    Two workgroups of 8 per CU at 128 registers where the LDS holds two and a wavefront's sums
    stay in registers (53 species / 325 reactions: one workgroup per CU of 4 wavefronts with all
    registers takes 1.3 % longer). Larger mechanisms have one workgroup per CU: 12 wavefronts of 168
    registers up to 52 sums (129 / 1,231: 8 of 256 registers take 4 % longer, 16 of 128, which
    spill, 22 %), else 8 of 256 up to 112 sums, with values from LDS kept for three reactions at a
    time instead of six (160 / 1,000, 108 sums: with four 2.4 % longer; 12 wavefronts would have 99
    sums for 168 registers; all before the order of the sums' rounds and the searched rows). The
    limits of 112 sums and of 80 for the shorter segments are set by that one mechanism and have no
    measurement on their far side; 100 species / 2,200 reactions (89 sums) takes the same shape."""
    fits = lambda p: lds_bytes(p['em'].N, p['rows'], p['waves'], p['tight']) <= LDS_MAX
    most = lambda p: max(len(s) for s in p['sums'])
    p8 = plan(t, info)
    if not fits(p8):
        return None
    if lds_bytes(p8['em'].N, p8['rows'], WAVES, p8['tight']) <= LDS_MAX // 2 and most(p8) <= 36:
        return p8, 4, SEGMENT
    p12 = plan(t, info, 12)
    if fits(p12) and most(p12) <= 52:
        return p12, 3, SEGMENT
    return (p8, 2, SEGMENT if most(p8) <= 80 else 3) if most(p8) <= 112 else None


def pays(t, info):
    """The shape if a mechanism's reactions are split, else None. A state's modelled load has to be
    worth the barriers and the per-wavefront prologue. 1,048,576 states, one wavefront per 64 states
    -> split, FP64 (mixed): load 7,000 (10 species / 15 reactions) 127 -> 191 us (77 -> 161), 8,700
    (10 / 22) 191 -> 216 (124 -> 194), 12,300 (11 / 30) 226 -> 264 (122 -> 213), 17,100 (12 / 40) 284
    -> 273 (223 -> 206), 24,000 (14 / 60) 457 -> 337 (478 -> 245), 42,100 (20 / 100) 2,061 -> 555
    (1,826 -> 370). The line lies at 16,000."""
    em = E._RateEmitter(t, info)
    if sum(reaction_cost(em, r) for r in range(em.R)) < 16000:
        return None
    return shape(t, info)


def emit(t, info, variant='fp64', shaped=None):
    p, occupancy, segment = shaped or shape(t, info)
    hot_rows = HOT_ROWS if segment == SEGMENT else None
    waves = p['waves']
    em = E._RateEmitter(t, info)
    runs = [order(em, rs, segment, hot_rows) for rs in p['rs']]
    N = em.N
    mixed = variant == 'mixed_valu'
    em.arrh32 = mixed
    name = f'kx_bk1_{variant}'
    lit = E._literal
    own = [[k for k in range(N) if k % waves == v] for v in range(waves)]
    per = max(len(o) for o in own)
    S = E._Src()
    # NASA-7: [piece: 0 = T > T_mid, 1 = T <= T_mid][species][14]: Gibbs in 0..6, enthalpy in 8..13
    PT = np.zeros((2, N, 14))
    for k in range(N):
        PT[0, k, :7], PT[0, k, 8:14] = t['g_hi'][k], t['h_hi'][k]
        PT[1, k, :7], PT[1, k, 8:14] = t['g_lo'][k], t['h_lo'][k]
    tab = lambda nm, a: S(f'__device__ const double {name}_{nm}[{len(a)}] __attribute__((aligned(16))) = {{' +
                          ', '.join(lit(v) for v in a) + '};', 0)
    tab('poly', PT.reshape(-1))
    tab('rcpW', list(t['rcpW']) + [0.0] * (waves * per - N))
    tab('tmid', t['T_mid'])
    S(RL._table(f'{name}_rrow', [p['rrow'].get(k, -1) for k in range(N)], 'int'), 0)
    S(RL._table(f'{name}_crow', [p['crow'].get(k, -1) for k in range(N)], 'int'), 0)
    plog = None
    if np.any(em.kind == M.PLOG):
        d = RL.plog_data(t)
        for nm, ct in (('plo', 'int'), ('plP', 'double'), ('pllnP', 'double'), ('plrcp', 'double'),
                       ('plko', 'int'), ('plnk', 'int'), ('plk', 'double')):
            S(RL._table(f'{name}_{nm}', d[nm], ct), 0)
        for line in RL.plog_helpers(name):
            S(line, 0)
        plog = lambda r: f'{name}_plog({r}, P, lnP, log2T, rcpT)'
    S(f'extern "C" __device__ const int {name}_lanes_per_state = {waves};', 0)
    S(f'extern "C" __global__ void __launch_bounds__({64 * waves}) '
      f'__attribute__((amdgpu_waves_per_eu({occupancy}, {occupancy})))', 0)
    S(f'{name}(const int n_states, const long long offsetT, const long long offset,', 0)
    S('            const double pressure_R, const double pressure_,', 0)
    S('            const double* __restrict__ state, double* __restrict__ rates, const double Tref)', 0)
    S('{', 0)
    staged, tight = not p['tight'], p['tight']
    if staged:
        S(f'__shared__ __attribute__((aligned(16))) double poly_s[{PT.size}];')
    S(f'__shared__ double rows[{p["rows"]} * {ROW}];        // w, rg, third-body C; then the wavefronts\' sums')
    if tight:
        S(f'double* const part = rows + {N * ROW};   // before rg is written and after the sums are read')
    else:
        S(f'__shared__ double part[{waves + 1} * {ROW}];')
    if staged:
        S(f'for (int i = threadIdx.x; i < {PT.size // 2}; i += {64 * waves})')
        S(f'  ((double2*)poly_s)[i] = ((const double2*){name}_poly)[i];')
    S('const int lane = threadIdx.x & 63;')
    S('const int v = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);      // part of the reactions')
    S(f'const long long first = (long long)blockIdx.x * {ROW};')
    S('const long long at = first + lane;')
    S('const bool live = at < n_states;')
    S('const long long id = live ? at : first;          // lanes past the end redo the first state, store nothing')
    S('const double T = Tref * state[id];')
    S('const double* const Y = state + id + offsetT;')
    S(f'double c[{per}];')
    S('double sum = 0.0;')
    S('#pragma unroll')
    S(f'for (int i = 0; i < {per}; ++i) {{')
    S(f'  c[i] = Y[min(v + {waves} * i, {N - 1}) * offset];             // every load in flight before the first use')
    S('}')
    S('#pragma unroll')
    S(f'for (int i = 0; i < {per}; ++i) {{')
    S(f'  c[i] = fmax(0.0, c[i]) * {name}_rcpW[v + {waves} * i];          // 0 past the last species')
    S('  sum += c[i];')
    S(f'  if (v + {waves} * i < {N}) rows[(v + {waves} * i) * {ROW} + lane] = c[i];   // for the loop over species')
    S('}')
    S(f'part[v * {ROW} + lane] = sum;')
    S(f'if (v == {waves - 1}) part[{waves} * {ROW} + lane] = log(T);   // once per state')
    S('const double rcpT = 1.0 / T;')
    S('const double T2 = T * T, T3 = T * T * T, T4 = T * T * T * T;')
    S('const double rcpT2 = rcpT * rcpT;')
    S('__syncthreads();')
    S('double rcpMbar = 0.0;')
    S('#pragma unroll')
    S(f'for (int i = 0; i < {waves}; ++i) rcpMbar += part[i * {ROW} + lane];')
    S(f'const double lnT = part[{waves} * {ROW} + lane];')
    if tight:
        S('__syncthreads();')
    S('const double omlnT = 1.0 - lnT;')
    S('const double log2T = lnT * 1.4426950408889634;')
    S('const float Tf = (float)T, rcpTf = (float)rcpT, log2Tf = (float)log2T;')
    S('const double P = pressure_, lnP = log(P);   // PLOG reactions (uniform per launch)')
    S('(void)P; (void)lnP; (void)log2T; (void)rcpT2; (void)Tf; (void)rcpTf; (void)log2Tf;')
    S('const double rho = pressure_R * rcpT / rcpMbar;')
    S('const double Cm = rho * rcpMbar;')
    S(f'const double C0 = {lit(float(t["one_atm_R"]))} * rcpT;')
    S(f'const double rcpC0 = {lit(float(t["R_one_atm"]))} * T;')
    S('// ---- species: w_k = C_k exp(g_k), rg_k = exp(-g_k), third-body concentrations')
    S('// (a loop: the exponential\'s constants stay in registers; unrolled they were moved there for')
    S('// each species, a third of the phase\'s vector instructions)')
    S(f'const double* const piece = {"poly_s" if staged else name + "_poly"};')
    S('#pragma unroll 1')
    S(f'for (int k = v; k < {N}; k += {waves}) {{')
    S(f'  const int rr = {name}_rrow[k], cr = {name}_crow[k];')
    S(f'  const double ck = rows[k * {ROW} + lane] * rho;')
    S(f'  const double* a = piece + 14 * k + (T > {name}_tmid[k] ? 0 : {14 * N});')
    S('  const double gk = a[0] * omlnT + a[1] * T + a[2] * T2 + a[3] * T3 + a[4] * T4 + a[5] * rcpT - a[6];')
    S('  const double ek = kx_exp(gk);')
    S(f'  rows[k * {ROW} + lane] = ck * ek;')
    S(f'  if (rr >= 0) rows[rr * {ROW} + lane] = kx_rcp(ek);')
    if p['crow']:
        S(f'  if (cr >= 0) rows[cr * {ROW} + lane] = ck;')
    S('  (void)cr;')
    S('}')
    S('__syncthreads();')
    S('// ---- reactions of each wavefront')
    mx = max(len(s) for s in p['sums'])
    S(f'double wd[{mx}];')
    S('#pragma unroll')
    S(f'for (int i = 0; i < {mx}; ++i) wd[i] = 0.0;')
    S('int o = lane;                                     // made opaque between segments')
    sets, sidx = em.efficiency_sets()
    at = lambda row: f'rows[{row * ROW} + o]'
    conc = lambda k: at(p['crow'][k]) if k in p['crow'] else f'({at(p["wrow"][k])} * {at(p["rrow"][k])})'
    for w in range(waves):
        S(f'{"if" if w == 0 else "else if"} (v == {w}) {{' if w < waves - 1 else 'else {')
        slot = {k: i for i, k in enumerate(p['sums'][w])}
        have_third, pins = set(), []
        run, hot = runs[w]
        for x, k in sorted(hot):
            S(f'const double hot_{x}{k} = {at(p["wrow" if x == "w" else "rrow"][k])};')
        row = lambda x, k: f'hot_{x}{k}' if (x, k) in hot else at(p['wrow' if x == 'w' else 'rrow'][k])
        for n, r in enumerate(run):
            if n % segment == 0:
                # the segment's sums are needed as values here: the compiler otherwise defers
                # them to the end of the wavefront's program, all values read from LDS alive
                S(f'asm volatile("" : "+v"(o){"".join(f", {q}" for q in pins)});')
                S('__builtin_amdgcn_sched_barrier(0);')
                pins = []
            # third body of this reaction, once per wavefront
            need = None
            if em.kind[r] not in (M.ELEMENTARY, M.PLOG):
                need = em._third_w(r, sidx)
            if need and need != 'Cm' and need not in have_third:
                have_third.add(need)
                if need.startswith('eff'):
                    terms = ['Cm']
                    for k, e in enumerate(sets[int(need[3:])]):
                        if e != 1.0:
                            terms.append(f'+ {lit(e - 1.0)} * {conc(k)}')
                    S(f'const double {need} = ' + ' '.join(terms) + ';')
                else:
                    S(f'const double {need} = {conc(int(need[1:]))};')
            ks = sorted({int(k) for k in np.flatnonzero((em.nu_f[r] > 0) | (em.rev[r] & (em.nu_r[r] > 0)))})
            S(f'double q{r};')
            S('{')
            for k in ks:
                S(f'const double W{k} = {row("w", k)};')
            for k in np.flatnonzero(em.nu_f[r]):
                S(f'const double rg{k} = {row("rg", int(k))};')
            T_ = E._Src()
            em.emit_reaction_p(T_, r, sidx, wvar='W', declare=False, plog=plog)
            for line in T_.lines:
                S.lines.append('  ' + line)
            S('}')
            for k in np.flatnonzero(em.net[r]):
                nu = int(em.net[r, k])
                term = f'q{r}' if abs(nu) == 1 else f'{lit(abs(nu))} * q{r}'
                i = slot[int(k)]
                if f'"+v"(wd[{i}])' not in pins:
                    pins.append(f'"+v"(wd[{i}])')
                S(f'wd[{i}] {"+=" if nu > 0 else "-="} {term};')
        S('__builtin_amdgcn_sched_barrier(0);')
        S('}')
    S('// ---- the wavefronts\' sums meet in LDS, added by the species\' owners in wavefront order')
    S(f'double acc[{per}];')
    S('#pragma unroll')
    S(f'for (int i = 0; i < {per}; ++i) acc[i] = 0.0;')
    for rnd in p['rounds']:
        S('__syncthreads();')
        for w in sorted({w for w, _ in rnd}):
            S(f'if (v == {w}) {{')
            for i, k in enumerate(p['sums'][w]):
                if (w, k) in rnd:
                    S(f'  rows[{rnd[(w, k)] * ROW} + lane] = wd[{i}];')
            S('}')
        S('__syncthreads();')
        for v in range(waves):
            S(f'{"if" if v == 0 else "else if"} (v == {v}) {{')
            for i, k in enumerate(own[v]):
                for w in range(waves):
                    if (w, k) in rnd:
                        S(f'  acc[{i}] += rows[{rnd[(w, k)] * ROW} + lane];')
            S('}')
    S('// ---- heat release rate and mass production rates; the stores last, so that no table load waits')
    S('// behind them; where registers are short powers of T again instead of held over the reactions')
    S('double Te = T, sh = 0.0;')
    if tight:
        S('asm volatile("" : "+v"(Te));')
    S('const double Te2 = Te * Te, Te3 = Te * Te * Te, Te4 = Te * Te * Te * Te;')
    W = t['W']
    for v in range(waves):
        S(f'{"if" if v == 0 else "else if"} (v == {v}) {{')
        for i, k in enumerate(own[v]):
            if k in em.active:
                S(f'  {{ const double* a = piece + {14 * k + 8} + (T > {lit(float(t["T_mid"][k]))} ? 0 : {14 * N});')
                S(f'    sh += acc[{i}] * (a[0] + a[1] * Te + a[2] * Te2 + a[3] * Te3 + a[4] * Te4 + a[5] * rcpT); }}')
        S('}')
    if tight:
        S('__syncthreads();                       // the last round\'s rows read by all')
    S(f'part[v * {ROW} + lane] = sh;')
    S('__syncthreads();')
    for v in range(waves):
        S(f'{"if" if v == 0 else "else if"} (v == {v}) {{')
        S('  if (live) {')
        for i, k in enumerate(own[v]):
            val = f'{lit(W[k])} * acc[{i}]' if k in em.active else '0.0'
            S(f'    rates[id + offsetT + {k} * offset] = {val};')
        S('  }')
        S('}')
    S('if (v == 0 && live) {')
    S('  double sum_h = 0.0;')
    S('  #pragma unroll')
    S(f'  for (int i = 0; i < {waves}; ++i) sum_h += part[i * {ROW} + lane];')
    S(f'  rates[id] = {lit(-float(t["R"]))} * T * sum_h;')
    S('}')
    S('}', 0)
    return S.text()
