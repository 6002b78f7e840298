"""Calls of mixed lengths with graphs: a call of up to 16 steps is replayed whatever
was captured before it, the rest of a longer one past its graphs of 16 is launched
singly, and the state is that of eager steps, bit for bit."""
import numpy as np
import pytest

from sunset_amd.nodes import jittered_lattice, taylor_green_ic

pytestmark = pytest.mark.gpu

PH = dict(Re=1.0, Wi=1.0, beta=0.5, eps=0.1, Ma=0.1)


@pytest.mark.parametrize("form,nx", [("di", 20), ("lc", 182)])   # 6 and 8 launches a step
def test_mixed_lengths(form, nx):
    import sunset_amd
    print(f"[graph lengths] {form} {nx}", flush=True)
    ns = jittered_lattice(nx, nx - 1, seed=nx, h_over_s=1.8, box=(0.0, 1.0, 0.0, (nx - 1) / nx))
    ic = taylor_green_ic(ns)
    pair = []
    for _ in range(2):
        s = sunset_amd.Solver(morder=4, form=form).setup(ns)
        s.set_phys(**PH)
        s.set_initial(ic, dt=1e-6, itime=3)
        pair.append(s)
    g, e = pair

    def same():
        a, b = g.fields(), e.fields()
        assert np.isfinite(a["ro"]).all()
        for k in ("ro", "rou", "rov", "cxx", "cxy", "cyy", "dt", "time", "itime"):
            assert np.array_equal(a[k], b[k]), k
    for rounds in range(2):
        for n in (1, 16, 3, 10, 1, 31, 33, 15, 0, 20, 2):
            g.run(n, graph=True)
            assert g.timing("graph_steps") == (n if n <= 16 else n // 16 * 16), n
            e.run(n)
            assert e.timing("graph_steps") == 0
            if rounds == 0:
                same()
        same()
        for s in pair:          # no graph of the old physics is replayed
            s.set_phys(**dict(PH, Wi=0.5, eps=0.3))
    for s in pair:
        s.close()
