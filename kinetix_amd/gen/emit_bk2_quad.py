"""FP64 transport with four lanes per state: kx_bk2_fp64, kx_bk2_fp64_pstate and the
surrogate's kx_bk2_fp64_queue on the wave-level routine of csrc/kx_bk2_quad.h.

This module builds the routine's table (one FP64 __device__ array per mechanism; each workgroup
stages it in LDS, the whole of it up to 72 species, else the species part, with the pair rows
streamed through two row buffers) and emits the kernels around it. With NB = ceil(N / 4) slots of four
species and one block (m, j) per slot pair j <= m, the table holds, in this order:

  rows m = 0 .. NB - 1, each fitA then fitC of its m + 1 blocks:
  fitA [block][64]   the diffusion fits' A operand of v_mfma_f64_16x16x4_f64: lane l holds the
                     coefficient of t^(l / 16 + 1) of the pair in row l % 16; row 4 c + g is
                     the pair (4 m + c, 4 j + g)
  fitC [block][g][c] their constant terms, in the accumulator's layout (element c of lane group g)
  wilT [slot][rank block][64], wil [16 species][rank group][64]
                     the factor L of M_kj = (8 (W_k + W_j))^(-1/2) = (L L^T)_kj (wilke_factor) as
                     A operands of L^T v (row l % 16: rank, k = l / 16: species 4 m + k) and of
                     L z (rows as visc, k: rank 4 q + l / 16)
  visc, cond         per 16 species (slots 4 h .. 4 h + 3): A operands [h][64] and constants
                     [h][g][c]; row 4 c + g is species 4 (4 h + c) + g. The viscosity fits are
                     scaled by W^(-1/4) (u = eta W^(-1/4))
  1/W, W, sqrt(W)    [species]

All fits are polynomials in t = ln T - t0, with t0 the middle of the fit window, expanded
exactly (rational arithmetic) from those in ln T and rounded once. Rows of pairs k = j and of
padding species (k >= N) evaluate to 1 and carry no weight.
"""
from __future__ import annotations

import math
from decimal import Decimal, getcontext
from fractions import Fraction

import numpy as np

from . import emit_hip as E

LDS_MAX = 160 * 1024
LPS = 4                      # lanes per state
WAVES = 8                    # wavefronts per workgroup: two per SIMD, up to 256 VGPRs each


def slots(N):
    return (N + 3) // 4


def wilke_factor(W):
    """L (N x r) with (L L^T)_kj = (8 (W_k + W_j))^(-1/2) to FP64 rounding: pivoted Cholesky in 50
    digits until the residual is 1e-16 of every diagonal entry, rounded once at the end (the
    entries of the product are within 1e-15 of the matrix for the mechanisms here)."""
    prec, getcontext().prec = getcontext().prec, 50
    try:
        w = [Decimal(float(v)) for v in W]
        n = len(w)
        entry = lambda k, j: 1 / (8 * (w[k] + w[j])).sqrt()
        d0 = [entry(k, k) for k in range(n)]
        d, L = list(d0), []
        while len(L) < n:
            p = max(range(n), key=lambda k: d[k] / d0[k])
            if d[p] < d0[p] * Decimal('1e-16'):
                break
            s = d[p].sqrt()
            col = [(entry(k, p) - sum(c[k] * c[p] for c in L)) / s for k in range(n)]
            L.append(col)
            d = [max(Decimal(0), a - c * c) for a, c in zip(d, col)]
        return np.array([[float(v) for v in col] for col in L]).T
    finally:
        getcontext().prec = prec


def rank_groups(t):
    """KR: groups of four ranks of the Wilke factor."""
    return (wilke_factor(np.asarray(t['W'])).shape[1] + 3) // 4


def table_doubles(N, kr):
    nb = slots(N)
    sg, blk, rb = (nb + 3) // 4, nb * (nb + 1) // 2, (kr + 3) // 4
    n = 80 * blk + 64 * nb * rb + 64 * sg * kr + 160 * sg + 12 * nb
    return (n + 1) & ~1


def row_doubles(N):
    """The pair rows, and the longest of them."""
    nb = slots(N)
    return 40 * nb * (nb + 1), 80 * nb


def lds_bytes(t, staged=False):
    N = int(t['n_species'])
    rows, longest = row_doubles(N)
    n = table_doubles(N, rank_groups(t))
    return 8 * (n - rows + 2 * longest if staged else n)


def center(t):
    """t0: the middle of the fit window in ln T (a multiple of 1/16: exact in FP64)."""
    lo, hi = float(np.min(t['T_fit'])), float(np.max(t['T_fit']))
    return round(16 * 0.5 * (math.log(lo) + math.log(hi))) / 16


def shifted(c, t0):
    """Coefficients of sum_i c_i x^i in powers of x - t0, exact before one rounding each."""
    c = [Fraction(float(v)) for v in c]
    s = Fraction(t0)
    return [float(sum(c[i] * math.comb(i, k) * s ** (i - k) for i in range(k, len(c))))
            for k in range(len(c))]


def table(t):
    N = int(t['n_species'])
    nb = slots(N)
    sg, blk = (nb + 3) // 4, nb * (nb + 1) // 2
    t0 = center(t)
    W = np.asarray(t['W'], dtype=np.float64)
    one = [1.0, 0.0, 0.0, 0.0, 0.0]
    fit = {(k, j): shifted(t['diff'][k, j], t0) for k in range(N) for j in range(k)}
    fit.update({(j, k): v for (k, j), v in list(fit.items())})
    fitA, fitC = np.zeros((blk, 64)), np.ones((blk, 4, 4))
    for m in range(nb):
        for j in range(m + 1):
            b = m * (m + 1) // 2 + j
            for c in range(4):
                for g in range(4):
                    k, i = 4 * m + c, 4 * j + g
                    f = fit.get((k, i), one)
                    fitC[b, g, c] = f[0]
                    for q in range(4):
                        fitA[b, 16 * q + 4 * c + g] = f[q + 1]
    Lw = wilke_factor(W)
    kr = (Lw.shape[1] + 3) // 4
    rb = (kr + 3) // 4
    L = np.zeros((16 * sg, 16 * rb))
    L[:N, :Lw.shape[1]] = Lw
    wilT, wil = np.zeros((nb, rb, 64)), np.zeros((sg, kr, 64))
    for l in range(64):
        i, q = l % 16, l // 16
        for m in range(nb):
            for h in range(rb):
                wilT[m, h, l] = L[4 * m + q, 16 * h + i]
        for h in range(sg):
            for r in range(kr):
                wil[h, r, l] = L[4 * (4 * h + i // 4) + i % 4, 4 * r + q]

    def species(coef, scale):
        A, C = np.zeros((sg, 64)), np.ones((sg, 4, 4))
        for h in range(sg):
            for c in range(4):
                for g in range(4):
                    k = 4 * (4 * h + c) + g
                    if k < N:
                        f = [v * scale[k] for v in shifted(coef[k], t0)]
                        C[h, g, c] = f[0]
                        for q in range(4):
                            A[h, 16 * q + 4 * c + g] = f[q + 1]
        return [A, C]
    pad = lambda v: np.concatenate([v, np.zeros(4 * nb - N)])
    rows = [v[m * (m + 1) // 2:(m + 1) * (m + 2) // 2] for m in range(nb) for v in (fitA, fitC)]
    parts = rows + [wilT, wil] + species(t['visc'], [1.0 / math.sqrt(math.sqrt(w)) for w in W]) \
        + species(t['cond'], np.ones(N)) \
        + [pad(np.asarray(t['rcpW'], dtype=np.float64)), pad(W), pad(np.sqrt(W))]
    flat = np.concatenate([p.reshape(-1) for p in parts])
    return np.concatenate([flat, np.zeros(table_doubles(N, kr) - flat.size)])


def fits(t):
    """Whether a mechanism takes this family, with its whole table in LDS. N >= 20: below, the
    4-fold repeated per-state work (T powers, divides) and padding species outweigh the shared
    pairs. 1,048,576 states of subsets of GRI-3.0, one state per lane -> this: 16 species 208 -> 207
    us, 18 249 -> 289, 19 269 -> 290, 20 313 -> 292, 21 (three padding species) 343 -> 355, 22 381 ->
    345, 24 429 -> 347, 32 668 -> 483; 9 species 69 -> 144, 53 1,861 -> 910. Calls of 100,003 states
    and fewer are faster from 16 species on (20: 41 -> 35 us, 1,000 states 34 -> 10), and a line by
    calls would need both kernels in every code object. At the other end the table has to fit the 160
    KB of a CU's LDS (N <= 72)."""
    return int(t['n_species']) >= 20 and lds_bytes(t) <= LDS_MAX


def fits_staged(t):
    """Whether it does with the pair rows streamed through LDS: up to 160 species, whose 40 slots
    of x and of the sums take 160 of a wavefront's 256 VGPRs."""
    return 20 <= int(t['n_species']) <= 160 and lds_bytes(t, True) <= LDS_MAX


def emit(t, info, waves=WAVES, staged=False, mfma=True):
    """kx_bk2_fp64, kx_bk2_fp64_pstate, beside straight-line kernels also kx_bk2_fp64_mfma (the
    transport entry point that asks for the Wilke sum on FP64 MFMA: the same kernel here), and
    with the table resident (every mechanism a surrogate can have) kx_bk2_fp64_queue."""
    N = int(t['n_species'])
    rcp = 'true' if int(t.get('rcp_diff', 0)) else 'false'
    kr = rank_groups(t)
    n = table_doubles(N, kr)
    rows, longest = row_doubles(N)
    t0, rcpR = repr(center(t)), E._literal(1.0 / float(t['R']))
    S = E._Src()
    S('#include "kx_bk2_quad.h"   // four lanes per state (kinetix_amd/csrc)', 0)
    S(f'__device__ const double kx_bk2_tab[{n}] __attribute__((aligned(16))) = {{' +
      ', '.join(E._literal(v) for v in table(t)) + '};', 0)
    if staged:
        tab = [f'__shared__ __attribute__((aligned(16))) double tab[{n - rows}], rows[{2 * longest}];',
               f'kxquad::stage<{n - rows}, {64 * waves}>(tab, kx_bk2_tab + {rows});']
        args = 'tab, rows, kx_bk2_tab'
    else:
        tab = [f'__shared__ __attribute__((aligned(16))) double rows[{n}];',
               f'kxquad::stage<{n}, {64 * waves}>(rows, kx_bk2_tab);']
        args = f'rows + {rows}, rows, nullptr'
    forms = [('kx_bk2_fp64', False), ('kx_bk2_fp64_mfma', False), ('kx_bk2_fp64_pstate', True)]
    for name, ps in forms if mfma else forms[::2]:
        S(f'extern "C" __device__ const int {name}_states_per_group = 16;', 0)
        S(f'extern "C" __global__ void __launch_bounds__({64 * waves})', 0)
        S(f'{name}(const int n_states, const long long offsetT, const long long offset,', 0)
        S('            ' + ('const double* __restrict__ p_state,' if ps else 'const double pressure,'), 0)
        S('            const double* __restrict__ state, double* __restrict__ conductivity,', 0)
        S('            double* __restrict__ viscosity, double* __restrict__ rhoD,', 0)
        S('            ' + ('double* __restrict__ Dkm, ' if ps else '') + 'const double Tref,', 0)
        S('            const int* __restrict__ n_dev)', 0)
        S('{', 0)
        S('// n_dev (optional): a state count known only on the device')
        S('const long long n_eff = n_dev ? min((long long)n_states, (long long)max(*n_dev, 0)) : (long long)n_states;')
        S('if (16ll * blockIdx.x >= n_eff) return;        // whole workgroup past the end')
        for line in tab:
            S(line)
        S(f'kxquad::plain<{N}, {kr}, {rcp}, {waves}, {"true" if ps else "false"}, {"true" if staged else "false"}>(')
        S(f'    {args}, n_eff, offsetT, offset, ' + ('p_state, 0.0' if ps else 'nullptr, pressure') +
          ', state, conductivity, viscosity, rhoD,')
        S('    ' + ('Dkm' if ps else 'nullptr') + f', Tref, {t0}, {rcpR});')
        S('}', 0)
    if staged:
        return S.text()
    S('// the surrogate\'s plain pass over a device queue of state ids (kxquad::queued)', 0)
    S(f'extern "C" __device__ const int kx_bk2q_lanes = {LPS};', 0)
    S('extern "C" __device__ const int kx_bk2_fp64_queue_states_per_group = 16;', 0)
    S(f'extern "C" __global__ void __launch_bounds__({64 * waves})', 0)
    S('kx_bk2_fp64_queue(const int n_audit,', 0)
    S('            const int* __restrict__ queue, int* __restrict__ counters,', 0)
    S('            const int* __restrict__ flags, const double tol, const double tol_rhoD,', 0)
    S('            const long long offsetT, const long long offset,', 0)
    S('            const double* __restrict__ p_state,', 0)
    S('            const double* __restrict__ state, double* __restrict__ conductivity,', 0)
    S('            double* __restrict__ viscosity, double* __restrict__ rhoD,', 0)
    S('            double* __restrict__ Dkm, const double Tref)', 0)
    S('{', 0)
    S('const long long valid = (long long)n_audit + max(counters[0], 0);')
    S('if (16ll * blockIdx.x >= valid) return;           // whole workgroup past the queue')
    for line in tab:
        S(line)
    S(f'kxquad::queued<{N}, {kr}, {rcp}, {waves}>(rows + {rows}, rows, valid, n_audit, queue, counters, flags,')
    S(f'    tol, tol_rhoD, offsetT, offset, p_state, state, conductivity, viscosity, rhoD, Dkm, Tref, {t0}, {rcpR});')
    S('}', 0)
    return S.text()
