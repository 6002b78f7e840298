"""The device-pointer operators, with a slice's neighbour values staged in LDS
where every slice has few distinct neighbours, against the drop-in operators,
which gather the caller's ghost values from memory: with ghosts equal to their
parents, bit for bit the same (one order of the sums).  Node counts around a
slice, wide stencils, walls and mirror ghosts; a shuffled node order, whose
slices have too many neighbours to stage; and the three in turn on one context,
whose layouts are built again.  Its own process: torch is imported before the
library."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CODE = r'''
import ctypes as C, dataclasses, sys
import torch
sys.path.insert(0, "sunset-viscoelastic_amd")
import numpy as np
import sunset_amd
from sunset_amd.nodes import jittered_lattice, wall_channel
L = sunset_amd.lib()


def shuffled(ns):
    p = np.random.default_rng(0).permutation(ns.npfb)
    return dataclasses.replace(ns, **{k: getattr(ns, k)[p] for k in
                                      ("x", "y", "s", "h", "h_small", "node_type")})


def check(s, ns, tag):
    n = ns.npfb
    rng = np.random.default_rng(3)
    _, _, irel, _ = s.ghosts()
    fields = [rng.uniform(-1, 1, n) for _ in range(3)]
    full = [np.concatenate([f, f[irel]]) for f in fields]
    host = {0: s.gradient, 1: s.laplacian, 4: s.filtered_var}
    for op, fn in host.items():
        want = [np.asarray(fn(f)) for f in full]
        src = [torch.tensor(f, device="cuda") for f in fields]
        dst = [torch.full(((2 if op == 0 else 1) * n,), float("nan"), dtype=torch.float64,
                          device="cuda") for _ in fields]
        a = (C.c_void_p * 3)(*[t.data_ptr() for t in src])
        b = (C.c_void_p * 3)(*[t.data_ptr() for t in dst])
        rc = L.sv_apply_dev(s.h, op, 3, a, b, None)
        assert rc == 0, L.sv_last_error(s.h)
        torch.cuda.synchronize()
        for f in range(3):
            got = dst[f].cpu().numpy()
            assert np.isfinite(got).all() and np.array_equal(got, want[f].ravel()), (tag, op, f)


sets = [(jittered_lattice(8, 8, seed=1, h_over_s=1.3), 4),      # exactly one slice
        (jittered_lattice(13, 5, seed=1, h_over_s=1.0, box=(0, 1, 0, 5 / 13)), 4),   # one more
        (jittered_lattice(64, 48, seed=1, h_over_s=1.8, box=(0, 1, 0, 0.75)), 4),
        (jittered_lattice(65, 70, seed=1, h_over_s=2.7, box=(0, 1, 0, 70 / 65)), 8),
        (jittered_lattice(40, 40, seed=1, h_over_s=1.8, bc=(1, 1, 3, 3)), 4),
        (wall_channel(20, 20, order=6, seed=1), 6)]
for ns, order in sets:
    s = sunset_amd.Solver(morder=order, form="lc")
    plain = [ns] if ns.nb else [ns, shuffled(ns), ns]
    for k, q in enumerate(plain):
        s.setup(q)
        check(s, q, (ns.npfb, order, k))
        s.calc_weights(); s.calc_boundary_weights(); s.calc_sums(); s.filter_coefficients()
        check(s, q, (ns.npfb, order, k, "again"))
    s.close()
    print("done", ns.npfb, order, flush=True)
print("OK")
'''


def test_staged_operators_match_gathers():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", CODE], cwd=root, capture_output=True, text=True,
                       timeout=110)
    print(r.stdout[-2000:], r.stderr[-2000:], flush=True)
    assert r.returncode == 0 and "OK" in r.stdout
