"""sv_get_state at the node counts around which its copies are made together or one
by one, and for callers that ask for some of the fields: the same values, and
nothing written to the fields that a form does not have."""
import ctypes as C

import numpy as np
import pytest

from sunset_amd.nodes import jittered_lattice, taylor_green_ic

pytestmark = pytest.mark.gpu

KEYS = ("ro", "rou", "rov", "u", "v", "pxx", "pxy", "pyy", "cxx", "cxy", "cyy")


@pytest.mark.parametrize("form", ["lc", "di"])
@pytest.mark.parametrize("nx,ny", [(12, 11), (128, 128), (113, 145)])   # 16384, 16385
def test_all_and_some_fields(form, nx, ny):
    import sunset_amd
    print(f"[get state] {form} {nx}x{ny}", flush=True)
    ns = jittered_lattice(nx, ny, seed=nx, h_over_s=1.8, box=(0.0, 1.0, 0.0, ny / nx))
    ic = taylor_green_ic(ns)
    ic["cxx"] = 1.0 + 0.2 * np.sin(2 * np.pi * ns.x) ** 2
    ic["cxy"] = 0.1 * np.cos(2 * np.pi * ns.y)
    s = sunset_amd.Solver(morder=4, form=form).setup(ns)
    s.set_phys(Re=1.0, Wi=1.0, beta=0.5, eps=0.1, Ma=0.1)
    s.set_initial(ic, dt=1e-6, itime=3)

    def get(keys, handle=None):
        out = {k: np.full(ns.npfb, -7.0) for k in keys}
        p = [out[k].ctypes.data_as(C.POINTER(C.c_double)) if k in out else None for k in KEYS]
        if handle is None:
            s._ck(sunset_amd.lib().sv_get_state(s.h, *p))
        else:
            s._ck(sunset_amd.lib().sv_ensemble_get_state(handle, 0, *p))
        return out
    first = get(KEYS)            # the caller's values, in the caller's order
    assert np.array_equal(first["ro"], ic["ro"])
    for k in ("u", "v"):
        assert np.abs(first[k] - ic[k]).max() <= 4 * np.finfo(float).eps * np.abs(ic[k]).max()
    if form == "di":
        for k in ("cxx", "cxy", "cyy"):
            assert np.array_equal(first[k], ic[k]), k
    s.run(1)
    E = sunset_amd.Ensemble([s])
    whole = get(KEYS)
    none = () if form == "lc" else ("pxx", "pxy", "pyy")
    for k in KEYS:
        if k in none:
            assert (whole[k] == -7.0).all(), k
        else:
            assert np.isfinite(whole[k]).all() and (whole[k] != -7.0).all(), k
        assert np.array_equal(get([k])[k], whole[k]), k
    some = get(("rov", "pxy", "cxx", "cyy"))
    for k, v in some.items():
        assert np.array_equal(v, whole[k]), k
    member = get(KEYS, E.h)
    for k in KEYS:
        assert np.array_equal(member[k], whole[k]), k
    E.close()
    s.close()
