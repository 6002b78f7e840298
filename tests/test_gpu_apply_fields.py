"""The device-pointer operators on several fields in one call: the same results,
bit for bit, as one call per field, for every number of fields a launch can
hold and one more, and for chained fields (one's output the next one's input),
whose launches have to follow each other.  Its own process: torch is imported
before the library."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CODE = r'''
import ctypes as C, sys
import torch
sys.path.insert(0, "sunset-viscoelastic_amd")
import numpy as np
import sunset_amd
from sunset_amd.nodes import jittered_lattice, wall_channel
L = sunset_amd.lib()
for ns, order in ((jittered_lattice(25, 23, seed=4, h_over_s=1.8), 4),
                  (wall_channel(16, 16, order=6, seed=1), 6)):
    s = sunset_amd.Solver(morder=order, form="lc").setup(ns)
    n = ns.npfb
    rng = np.random.default_rng(3)
    def call(op, src, dst):
        a = (C.c_void_p * len(src))(*[t.data_ptr() for t in src])
        b = (C.c_void_p * len(dst))(*[t.data_ptr() for t in dst])
        rc = L.sv_apply_dev(s.h, op, len(src), a, b, None)
        assert rc == 0, L.sv_last_error(s.h)
    for op in range(7):
        m = 2 * n if op == 0 else n
        for nf in range(1, 6):
            src = [torch.tensor(rng.uniform(-1, 1, n), device="cuda") for _ in range(nf)]
            one = [torch.empty(m, dtype=torch.float64, device="cuda") for _ in range(nf)]
            all_ = [torch.full_like(t, float("nan")) for t in one]
            for f in range(nf):
                call(op, src[f:f + 1], one[f:f + 1])
            call(op, src, all_)
            assert all(torch.equal(x, y) for x, y in zip(one, all_)), (op, nf)
        if op:
            a, b, c = (torch.tensor(rng.uniform(-1, 1, n), device="cuda") for _ in range(3))
            b2, c2 = torch.empty_like(b), torch.empty_like(c)
            call(op, [a], [b2]); call(op, [b2], [c2])
            call(op, [a, b], [b, c])          # b is read after it is written
            assert torch.equal(b, b2) and torch.equal(c, c2), ("chain", op)
    s.close()
print("OK")
'''


def test_fields_of_one_call():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", CODE], cwd=root, capture_output=True, text=True,
                       timeout=110)
    print(r.stdout[-2000:], r.stderr[-2000:], flush=True)
    assert r.returncode == 0 and "OK" in r.stdout
