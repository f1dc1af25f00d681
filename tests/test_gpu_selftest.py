"""The MFMA lane layout assumed by the generated mixed-precision kernels, checked on the
device against the host product of the same closed-form operands."""
import ctypes as C

import numpy as np
import pytest
import torch

from kinetix_amd.api import lib

pytestmark = pytest.mark.gpu


def test_mfma_f32_16x16x4_layout():
    L = lib()
    L.kx_selftest_mfma_layout.argtypes = [C.c_void_p, C.c_void_p]
    out = torch.full((256,), np.nan, dtype=torch.float32, device='cuda')
    assert L.kx_selftest_mfma_layout(C.c_void_p(out.data_ptr()), None) == 0
    torch.cuda.synchronize()
    A = np.array([[i + 16 * k + 1 for k in range(4)] for i in range(16)], dtype=np.float64)
    B = np.array([[(k + 1) * 100 + j for j in range(16)] for k in range(4)], dtype=np.float64)
    assert np.array_equal(out.cpu().numpy().reshape(16, 16).astype(np.float64), A @ B)


def _f64_probe(mode):
    L = lib()
    L.kx_selftest_mfma_f64_layout.argtypes = [C.c_int, C.c_void_p, C.c_void_p]
    out = torch.full((256,), np.nan, dtype=torch.float64, device='cuda')
    assert L.kx_selftest_mfma_f64_layout(mode, C.c_void_p(out.data_ptr()), None) == 0
    torch.cuda.synchronize()
    return out.cpu().numpy().reshape(64, 4)


def _raw(D):
    """D (16x16) in the FP64 result layout: lane l, element r = D[4 r + l // 16][l % 16]."""
    return np.array([[D[4 * r + l // 16, l % 16] for r in range(4)] for l in range(64)])


def test_mfma_f64_16x16x4_result_layout():
    """Every result entry names its own (row, column): D[i][j] = 16 i + j."""
    got = _f64_probe(1)
    D = np.array([[16.0 * i + j for j in range(16)] for i in range(16)])
    assert np.array_equal(got, _raw(D)), got


def test_mfma_f64_16x16x4_operand_layout():
    got = _f64_probe(0)
    A = np.array([[i + 16 * k + 1 for k in range(4)] for i in range(16)], dtype=np.float64)
    B = np.array([[(k + 1) * 100 + j for j in range(16)] for k in range(4)], dtype=np.float64)
    assert np.array_equal(got, _raw(A @ B))


def test_mfma_bf16_16x16x16_layout():
    L = lib()
    L.kx_selftest_mfma_bf16_layout.argtypes = [C.c_void_p, C.c_void_p]
    out = torch.full((256,), np.nan, dtype=torch.float32, device='cuda')
    assert L.kx_selftest_mfma_bf16_layout(C.c_void_p(out.data_ptr()), None) == 0
    torch.cuda.synchronize()
    A = np.array([[(i + 16 * k + 1) / 16.0 for k in range(16)] for i in range(16)])
    B = np.array([[(k + 1) * 3 + j for j in range(16)] for k in range(16)], dtype=np.float64)
    assert np.array_equal(out.cpu().numpy().reshape(16, 16).astype(np.float64), A @ B)


def test_mfma_bf16_16x16x32_layout():
    """The layout the surrogate's inference kernels (kx_mlp_wave.h) are built on."""
    L = lib()
    L.kx_selftest_mfma_bf16_k32_layout.argtypes = [C.c_void_p, C.c_void_p]
    out = torch.full((256,), np.nan, dtype=torch.float32, device='cuda')
    assert L.kx_selftest_mfma_bf16_k32_layout(C.c_void_p(out.data_ptr()), None) == 0
    torch.cuda.synchronize()
    A = np.array([[(i * 7 + k * 3) % 17 - 8 for k in range(32)] for i in range(16)], dtype=np.float64)
    B = np.array([[(k * 5 + j * 11) % 13 - 6 for j in range(16)] for k in range(32)], dtype=np.float64)
    assert np.array_equal(out.cpu().numpy().reshape(16, 16).astype(np.float64), A @ B)


def _rcp(y):
    L = lib()
    L.kx_selftest_rcp.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_void_p]
    d_in = torch.from_numpy(y).cuda()
    d_out = torch.full_like(d_in, np.nan)
    assert L.kx_selftest_rcp(y.size, C.c_void_p(d_in.data_ptr()), C.c_void_p(d_out.data_ptr()), None) == 0
    torch.cuda.synchronize()
    return d_out.cpu().numpy()


def test_refined_reciprocal_within_one_ulp():
    """kx_rcp, the reciprocal of the transport fits and of the rates' exp(g), 1 + Pr and Troe
    denominators: within 1 ulp of the exact 1/y over 600 decades of both signs, exact on powers
    of two."""
    rng = np.random.default_rng(20261202)
    y = 10.0 ** rng.uniform(-300, 300, 1 << 20)
    y[: 1 << 18] = rng.uniform(1e-6, 1e3, 1 << 18)            # the fits' own range
    y[1 << 18: 1 << 19] = 10.0 ** rng.uniform(-30, 30, 1 << 18)
    y[3 << 17: 5 << 17] *= -1.0
    pw = 2.0 ** np.arange(-1000, 1001)
    y = np.concatenate([y, pw, np.nextafter(pw, 0), np.nextafter(pw, np.inf), [1.0, 3.0, 0.1, 7.0]])
    r = _rcp(y)
    exact = 1.0 / y                                             # correctly rounded (IEEE)
    ulp = np.abs(r - exact) / np.spacing(np.abs(exact))
    assert np.all(np.isfinite(r)) and ulp.max() <= 1.0, ulp.max()
    assert np.array_equal(r[(1 << 20):(1 << 20) + pw.size], 1.0 / pw)


def _exp(which, x):
    L = lib()
    L.kx_selftest_exp.argtypes = [C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p]
    d_in = torch.from_numpy(np.ascontiguousarray(x, dtype=np.float64)).cuda()
    d_out = torch.full_like(d_in, 123.0)
    assert L.kx_selftest_exp(which, d_in.numel(), C.c_void_p(d_in.data_ptr()), C.c_void_p(d_out.data_ptr()), None) == 0
    torch.cuda.synchronize()
    return d_out.cpu().numpy()


def _ulp(got, exact):
    """Largest error in units in the last place of the exact (80-bit) values' FP64 rounding."""
    assert np.finfo(np.longdouble).nmant >= 63
    return float((np.abs(got.astype(np.longdouble) - exact) / np.spacing(np.abs(exact.astype(np.float64)))).max())


@pytest.mark.parametrize('which,f,lo,hi', [(0, np.exp2, -1021.0, 1023.5), (1, np.exp, -707.0, 709.5)])
def test_exponentials_within_an_ulp(which, f, lo, hi):
    """kx_exp2 and kx_exp over all exponents with a normal result, around 0 and around the points
    where the reduced argument changes sign; beyond them infinity or a result that is subnormal or
    zero, up to exponents that fill an int; a NaN stays one."""
    rng = np.random.default_rng(20261205)
    step = 1.0 if which == 0 else np.log(2.0)
    half = (np.arange(-1020, 1020) + 0.5) * step
    x = np.concatenate([rng.uniform(lo, hi, 1 << 20), rng.uniform(-2, 2, 1 << 18), 10.0 ** rng.uniform(-300, 0, 1 << 12),
                        half, np.nextafter(half, 0), np.arange(-1020, 1021) * step, [0.0, -0.0, lo, hi]])
    x = x[(x >= lo) & (x <= hi)]
    got = _exp(which, x)
    assert np.all(np.isfinite(got))
    assert _ulp(got, f(x.astype(np.longdouble))) <= 1.0
    assert np.all(got[x == 0.0] == 1.0)
    far = np.array([1025.0, 1100.0, 1e6, 2.0e9]) * step
    assert np.all(np.isposinf(_exp(which, far[:3]))) and np.all(_exp(which, -far[1:3]) == 0.0)
    if which == 0:
        assert np.isposinf(_exp(0, far[3:]))[0] and _exp(0, -far[3:])[0] == 0.0
    sub = rng.uniform(-1074.0, -1022.0, 4096) * step           # subnormal results: within their unit
    assert np.max(np.abs(_exp(which, sub).astype(np.longdouble) - f(sub.astype(np.longdouble)))) <= 2.0 ** -1074
    assert np.all(np.isnan(_exp(which, [np.nan])))


def test_log2_within_its_bound():
    """kx_log2 on normal numbers of every exponent and close to 1; exact on powers of two; NaN for 0,
    negative numbers and NaN. Relative error in units of 2^-53: m - 1 is exact, m + 1 rounded (1), its
    reciprocal within an ulp (2), their product s rounded (1), the polynomial's last fma (1), leading
    coefficient (1/2) and the rest (0.1, as s^2 < 0.03), and the last fma (1): 6.6, and no more with
    an exponent added, as the sum is then at least 1/2 and s p at most that."""
    rng = np.random.default_rng(20261206)
    pw = 2.0 ** np.arange(-1022, 1024)
    x = np.concatenate([2.0 ** rng.uniform(-1022, 1023.99, 1 << 20), rng.uniform(0.5, 2.0, 1 << 18),
                        1.0 + 10.0 ** rng.uniform(-15, -1, 1 << 16), 1.0 - 10.0 ** rng.uniform(-15, -1, 1 << 16),
                        np.sqrt(0.5) * pw[1:-1], np.nextafter(np.sqrt(0.5), 0) * pw[1:-1]])
    x = x[x != 1.0]
    got = _exp(2, x)
    assert np.all(np.isfinite(got))
    exact = np.log2(x.astype(np.longdouble))
    u = float(np.max(np.abs(got - exact) / np.abs(exact))) * 2.0 ** 53
    assert u <= 6.6, u
    assert np.array_equal(_exp(2, pw), np.arange(-1022.0, 1024.0))
    assert np.all(np.isnan(_exp(2, [0.0, -0.0, -1.0, -1e300, np.nan])))
