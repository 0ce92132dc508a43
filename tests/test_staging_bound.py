"""The device memory that calls keep for their transfers stays below 512 MB: fields
above that are staged in memory that is given back at the end of the call, fields
below it are not allocated for again.  On the host side of the library alone
(hip_stub.c), in a process of its own."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

from .test_out_of_memory import stub  # noqa: F401  (the fixture)

RUN = """
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_live.restype = ctypes.c_size_t
import numpy as np
from ntlp_amd import *
nx, ny, nz = eval(sys.argv[2])
s = DropletStep(Grid.uniform(nx, ny, nz, 0.02, 0.02, 0.02), Consts(), Flags())
f = np.zeros((nx, ny, nz + 2))
bare = stub.stub_live()
ext = (nx + 5) * (ny + 5) * (nz + 2)
s.set_fields(f, f, f, f, f)
held = stub.stub_live() - bare - ext * (5 * 8 + 3 * 4)
assert held == (f.nbytes if f.nbytes <= 512 << 20 else 0), held
s.step(MODE_BE, PREC_FP64, 1, 2)
bare = stub.stub_live()
s.wcell_counts()
s.calc_tauc_min()
assert stub.stub_live() - bare <= 512 << 20
"""


@pytest.mark.parametrize("dims", [(8, 6, 8), (256, 256, 128), (512, 512, 270)])
def test_what_is_kept(stub, dims):  # noqa: F811
    r = subprocess.run([sys.executable, "-c", RUN, stub, repr(dims)], cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       capture_output=True, text=True, timeout=240)
    assert r.returncode == 0, r.stderr[-2000:]
