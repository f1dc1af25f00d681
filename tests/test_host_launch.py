"""The host library's launches, on the CPU: its HIP calls bound to tests/hip_stub.c, in a process of
their own."""
import os
import subprocess
import sys

import pytest

from kinetix_amd import api

HERE = os.path.dirname(os.path.abspath(__file__))

LAUNCHES = '''
import ctypes as C, sys
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
L = C.CDLL(sys.argv[2])
n, block, lanes = (int(a) for a in sys.argv[3:])
C.c_int.in_dll(stub, 'stub_block').value = block
C.c_int.in_dll(stub, 'stub_lanes').value = lanes
meta = b'n_species 2\\nspecies A B\\nmolar_mass 0.002 0.032\\n'
h = C.c_int(0)
L.kx_last_error.restype = C.c_char_p
ok = lambda rc: rc == 0 or sys.exit(L.kx_last_error().decode())
ok(L.kx_init_image(meta, C.c_size_t(len(meta)), b'code', C.c_size_t(4), 0, C.byref(h)))
ok(L.kx_build(h, C.c_double(101325.0), C.c_double(1.0), (C.c_double * 2)(0.5, 0.5)))
S, R = 1 << 40, 1 << 50                      # addresses that nothing reads
ok(L.kx_production_rates(h, n, n, n, C.c_double(1.0), C.c_void_p(S), C.c_void_p(R), None))
class Launch(C.Structure):
    _fields_ = [('grid', C.c_uint), ('block', C.c_uint), ('n', C.c_int), ('state', C.c_void_p), ('rates', C.c_void_p)]
log = (Launch * 64).in_dll(stub, 'stub_log')
for i in range(C.c_int.in_dll(stub, 'stub_launches').value):
    l = log[i]
    print(l.grid, l.block, l.n, (l.state - S) // 8, (l.rates - R) // 8)
'''


@pytest.fixture(scope='module')
def stub(tmp_path_factory):
    out = str(tmp_path_factory.mktemp('stub') / 'hip_stub.so')
    subprocess.run(['gcc', '-O1', '-shared', '-fPIC', os.path.join(HERE, 'hip_stub.c'), '-o', out], check=True)
    return out


@pytest.mark.parametrize('n', [0, 1, 1000, 4194303, 4194304, (1 << 29) - 8, 1 << 29, (1 << 30) + 7, (1 << 31) - 1])
@pytest.mark.parametrize('block,lanes', [(256, 0), (512, 8), (768, 12), (1024, 32)])
def test_rates_of_any_state_count(stub, n, block, lanes):
    """Every state count an int holds is launched, whatever the kernel's lanes per state: pieces in
    order without gap or overlap, each a grid below 2^32 threads that covers its states, whole
    workgroups but the last."""
    if not os.path.exists(api.LIB_PATH):
        pytest.skip('libkinetix_mi.so not built (python -m kinetix_amd.build)')
    r = subprocess.run([sys.executable, '-c', LAUNCHES, stub, api.LIB_PATH, str(n), str(block), str(lanes)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    got = [[int(v) for v in line.split()] for line in r.stdout.splitlines()]
    per = block // max(lanes, 1)                      # states of a workgroup
    assert len(got) == -(-n // ((2 ** 32 - 1) // block * per))
    at = 0
    for grid, b, m, s, w in got:
        assert b == block and (s, w) == (at, at)
        assert grid == -(-m // per) and grid * b < 2 ** 32
        at += m
        assert m % per == 0 or at == n
    assert at == n
