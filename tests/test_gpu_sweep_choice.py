"""Which form of the halo-staged sweeps a node set gets (choose_blocks in
k_loop.hip), and the form that no compact node order reaches: 64 slots a workgroup
without the split by fields, where a larger set's 128- or 256-slot halos do not
fit.  Its fields equal the gathers' bit for bit, as every form's."""
import numpy as np
import pytest

from sunset_amd.nodes import jittered_lattice, taylor_green_ic

pytestmark = pytest.mark.gpu

PH = dict(Re=1.0, Wi=1.0, beta=0.5, eps=0.1, Ma=0.1)
FIELDS = ("ro", "rou", "rov", "cxx", "cxy", "cyy", "dt", "emax_np1")


def _set(nx, ny, order, **kw):
    ns = jittered_lattice(nx, ny, seed=nx, h_over_s={4: 1.8, 6: 2.4}[order],
                          box=(0.0, 1.0, 0.0, ny / nx), **kw)
    ic = taylor_green_ic(ns)
    ic["cxx"] = 1.0 + 0.2 * np.sin(2 * np.pi * ns.x) ** 2
    ic["cxy"] = 0.1 * np.cos(2 * np.pi * ns.y)
    return ns, ic


def _solver(ns, ic, order, form, mdiff=0.0, **options):
    import sunset_amd
    s = sunset_amd.Solver(morder=order, form=form)
    for k, v in options.items():
        s.set_option(k, v)
    s.setup(ns)
    s.set_phys(**PH, Mdiff=mdiff)
    s.set_initial(ic, dt=1e-6, itime=3)
    return s


def _form(s):
    return tuple(int(s.timing("sweep_" + k)) for k in ("slots", "fields", "stream"))


@pytest.mark.parametrize("nx,ny,order,form", [
    (33, 31, 4, (64, 1, 0)),
    (181, 181, 6, (64, 1, 0)),       # 32761 nodes
    (182, 181, 6, (128, 0, 0)),      # 32942
    (512, 499, 4, (128, 0, 1)),      # past 256 MB of weights
    (709, 707, 4, (256, 0, 1)),      # past 500k nodes
])
def test_form_by_size(nx, ny, order, form):
    print(f"[sweep choice] {nx}x{ny} order {order}", flush=True)
    ns, ic = _set(nx, ny, order)
    s = _solver(ns, ic, order, "di")
    assert _form(s) == form
    s.close()


@pytest.mark.parametrize("order,form,mdiff", [(6, "lc", 0.0), (6, "di", 1e-3), (4, "lc", 0.0),
                                              (4, "di", 0.0)])
def test_row_order_past_the_split(order, form, mdiff):
    """32942 nodes in rows of 181: halos of 128 slots have over a thousand records"""
    print(f"[sweep choice] rows, order {order} {form}", flush=True)
    ns, ic = _set(182, 181, order)
    out = []
    for halo in (0, 1):
        s = _solver(ns, ic, order, form, mdiff, loop_order=0, halo_sweeps=halo)
        assert _form(s) == ((64, 0, 0) if halo else (0, 0, 0))
        s.run(2)
        out.append(s.fields())
        s.close()
    for k in FIELDS:
        assert np.isfinite(out[0][k]).all() and np.array_equal(out[0][k], out[1][k]), k


def test_ensemble_of_row_ordered_members():
    """two members of 64-slot halos, together past the 128-slot line"""
    import sunset_amd
    print("[sweep choice] ensemble", flush=True)
    members = []
    for nx, ny in ((151, 149), (149, 140)):
        ns, ic = _set(nx, ny, 6)
        s = _solver(ns, ic, 6, "lc", loop_order=0)
        assert _form(s) == (64, 1, 0)
        members.append(s)
    E = sunset_amd.Ensemble(members)
    assert _form(E) == (64, 0, 0)
    E.run(2)
    for m, s in enumerate(members):
        s.run(2)
        a, b = E.fields(m), s.fields()
        for k in FIELDS:
            assert np.isfinite(b[k]).all() and np.array_equal(a[k], b[k]), (m, k)
    E.close()
    for s in members:
        s.close()
