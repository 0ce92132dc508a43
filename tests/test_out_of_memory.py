"""Device memory that runs out, on the host side of the library alone
(hip_stub.c): droplets on the device can be read back without any more of it, a
put needs no more than its droplets, and a call that cannot have its memory
leaves a context without droplets that refuses to step until they are put again.
Each case runs in a process of its own, before which the real runtime is not
loaded."""
from __future__ import annotations

import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_live.restype = ctypes.c_size_t
stub.stub_limit.argtypes = [ctypes.c_size_t]
import numpy as np
from ntlp_amd import *
N = int(sys.argv[2])

def context(nx=8, ny=6, nz=8):
    s = DropletStep(Grid.uniform(nx, ny, nz, 0.02, 0.02, 0.02), Consts(), Flags())
    f = np.zeros((nx, ny, nz + 2))
    s.set_fields(f, f, f, f + 300, f)
    return s

def code(call, *args):
    try:
        call(*args)
    except NtlpError as e:
        return e.code
    return 0

def droplets(n):
    p = Particles.empty(n)
    p.soa[:] = np.arange(1.0, 1 + p.soa.size).reshape(p.soa.shape)
    return p

def count(s):
    return s.lib.ntlp_gpu_particles_count()

NOMEM, STATE = -4, -7
s = context()
base = stub.stub_live()
s.generate(Ensemble(), N)
need = stub.stub_live() - base  # of N droplets, no more: one ensemble takes no staging
base -= 8 * 6 * 10 * 8  # without what set_fields staged
s.close()
assert stub.stub_live() == 0
s = context()
"""

CASES = {
    "transfers_need_no_memory_of_their_own": """
stub.stub_limit(base + need)
s.put(droplets(N))
ens = [Ensemble(seed=1), Ensemble(seed=2)]
for call in (s.get, s.get_records, lambda: s.column("x"), lambda: s.column("ufx"),
             lambda: s.put_records(np.zeros(352 * N, np.uint8)), s.get,
             lambda: s.generate(ens, [1, N - 1]), s.get, lambda: s.step(MODE_BE, PREC_FP64, 1, 2), s.get_records):
    call()
    assert count(s) == N
""",
    "droplets_that_do_not_fit": """
s.close()
for way in (lambda n: s.put(droplets(n)), lambda n: s.put_records(np.zeros(352 * n, np.uint8)),
            lambda n: s.generate(Ensemble(), n)):
    for first in (0, N // 2):
        for k in range(1, 32):  # each of the buffers is the one that fails
            stub.stub_limit(1 << 40)
            s = context()
            s.put(droplets(first))
            stub.stub_limit(base + need * k // 32)
            rc = code(way, N)
            assert rc == NOMEM, (rc, first, k, need, stub.stub_live() - base)
            assert count(s) == 0
            launches, s.n = stub.stub_launches(), 0
            for call in (lambda: s.step(MODE_BE, PREC_FP64, 1, 2), lambda: s.interp(True, True), s.get, s.get_records,
                         lambda: s.particle_update_rk3(1), s.calc_tauc_min, s.particle_xy_stats):
                assert code(call) == STATE
            assert stub.stub_launches() == launches
            stub.stub_limit(base + need)
            way(N)
            assert count(s) == N
            s.step(MODE_BE, PREC_FP64, 1, 2)
            s.close()
""",
    "an_empty_put_after_a_failed_one": """
stub.stub_limit(base + need // 2)
assert code(s.put, droplets(N)) == NOMEM
s.put(droplets(0))
s.step(MODE_BE, PREC_FP64, 1, 2)
assert count(s) == 0
""",
    "a_rejected_call_keeps_the_droplets": """
s.put(droplets(N))
assert code(s.generate, [Ensemble(mult=0)], [3]) == -1 and code(s.generate, [Ensemble()], [0]) == -5
assert s.lib.ntlp_gpu_particles_put(None, None, None, None, 5) == -1
assert count(s) == N
s.n = N
s.step(MODE_BE, PREC_FP64, 1, 2)
""",
    "staging_gives_way_to_droplets": """
s.put(droplets(1))
s.close()
s = context(64, 64, 30)
f = np.zeros((64, 64, 32))
live = stub.stub_live()
s.step(MODE_BE, PREC_FP64, 1, 2)
s.particle_coupling_exchange()
s.apply_particle_coupling(f.copy(), f.copy(), LAYOUT_CORE)  # stages two fields
n = N * 2 * f.nbytes // (2 * need)  # droplets of half of that
stub.stub_limit(stub.stub_live() + 1000)
s.put(droplets(n))
assert count(s) == n
s.get()
""",
}


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    so = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    subprocess.run([cc, "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "hip_stub.c")], check=True)
    return so


@pytest.mark.parametrize("n", [2, 1000, 40_000])
@pytest.mark.parametrize("case", CASES)
def test_memory(stub, case, n):
    r = subprocess.run([sys.executable, "-c", PRELUDE + CASES[case], stub, str(n)], cwd=os.path.dirname(HERE),
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
