"""Mirror ghosts need the halo sweeps, so the largest halos that are taken decide
which mirror sets run: 853 records of 64 slots, either form, are taken; more are
refused with that limit."""
import dataclasses

import numpy as np
import pytest

import oracle_lib as OL
from parity_util import FIELD_RTOL, field_rel
from sunset_amd.nodes import jittered_lattice

pytestmark = pytest.mark.gpu

PH = dict(Re=10.0, Wi=0.5, beta=0.5, eps=0.1, Ma=0.1)
STEPS, DT = 3, 1e-6


def _nodes(nx, ny, hos):
    """Symmetric on all edges: a slot may be read as itself and mirrored in x, in y
    and in both, four records a slot at most."""
    ns = jittered_lattice(nx, ny, seed=5, h_over_s=hos, bc=(2, 2, 2, 2),
                          box=(0.0, 1.0, 0.0, ny / nx))
    ns = dataclasses.replace(ns, smax=4 * ns.smax)      # the search cells follow smax
    x, y = ns.x, ns.y
    ic = dict(ro=1 + 0.01 * np.cos(2 * np.pi * x), u=0.1 * np.sin(np.pi * x), v=0 * x,
              cxx=1 + 0.05 * np.cos(np.pi * x) ** 2,
              cxy=0.02 * np.sin(np.pi * x) * np.sin(np.pi * y), cyy=np.ones(ns.npfb))
    return ns, ic


def _solver(ns, form):
    import sunset_amd
    s = sunset_amd.Solver(morder=4, form=form).setup(ns)
    s.set_phys(**PH)
    return s


@pytest.mark.parametrize("form", ["lc", "di"])
@pytest.mark.parametrize("hos,least", [(6.5, 800), (7.0, 820)])
def test_largest_mirror_halos_vs_oracle(form, hos, least):
    """210 nodes, 840 records in all: halos of up to 815 and 831 records"""
    print(f"[halo limit] {form} {hos}", flush=True)
    ns, ic = _nodes(15, 14, hos)
    s = _solver(ns, form)
    s.set_initial(ic, dt=DT, dt_mode="fixed")   # (the PID's error estimate of so smooth a
    #                                             state is rounding)
    # four slices, the last of 18 slots: the mean bounds the largest from below
    assert s.stencil_stats()["halo_per_node"] * ns.npfb / 4 > least - 50
    s.run(STEPS)
    F = s.fields()
    s.close()
    o = OL.OracleSim(ns, 4, nplink=900).setup()
    o.make_phys(form=form, dt_mode="fixed", **PH)
    o.set_initial(ic, dt=DT)
    o.run(STEPS)
    R = o.fields()
    assert F["dt"] == R["dt"] == DT
    keys = ("ro", "rou", "rov") + (("pxx", "pxy", "pyy") if form == "lc" else ("cxx", "cxy", "cyy"))
    for k in keys:
        assert np.isfinite(R[k]).all() and field_rel(F[k], R[k]) < FIELD_RTOL, k


@pytest.mark.parametrize("form", ["lc", "di"])
def test_larger_mirror_halos_are_refused(form):
    """240 nodes, all within each other's reach: 960 records"""
    import sunset_amd
    print(f"[halo limit] refused {form}", flush=True)
    ns, ic = _nodes(16, 15, 8.5)
    s = _solver(ns, form)
    with pytest.raises(sunset_amd.SunsetError, match="within 853 records"):
        s.set_initial(ic)
    s.close()
