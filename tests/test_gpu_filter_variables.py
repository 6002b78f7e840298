"""sv_filter_variables on six fields the caller holds (two launches, of four and
two fields): each filtered as the single-field operator does, bit for bit, on the
caller's own ghost values; rho then less its volume-weighted mean deviation."""
import ctypes as C

import numpy as np
import pytest

from sunset_amd.nodes import jittered_lattice, wall_channel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["ragged", "mirror", "walls"])
def test_filter_variables(kind):
    import sunset_amd
    print(f"[filter variables] {kind}", flush=True)
    order = 6 if kind == "walls" else 4
    ns = (wall_channel(16, 16, order=6, seed=1) if kind == "walls" else
          jittered_lattice(33, 31, seed=2, h_over_s=1.8,
                           bc=(2, 2, 1, 1) if kind == "mirror" else (1, 1, 1, 1)))
    s = sunset_amd.Solver(morder=order, form="di").setup(ns)
    n, npt = s.npfb, s.np
    assert npt > n
    rng = np.random.default_rng(7)
    f = [1.0 + 0.05 * rng.standard_normal(npt)] + [rng.standard_normal(npt) for _ in range(5)]
    want = [s.filtered_var(v).copy() for v in f]
    w = s.weights(s.stencil_stats()["K_max"])
    if kind != "walls":      # the operator by hand, ghost values included (a second search
        #                      would undo the pruning of boundary nodes' lists)
        o = sunset_amd.Solver(morder=order, form="di")
        o.set_nodes(ns)
        cnt, _, link = o.find_neighbours()
        o.close()
        K = link.shape[1]
        inside = np.arange(K) < cnt[:, None]
        for v, q in zip(f, want):
            g = np.where(inside, v[np.where(inside, link, 0)], 0.0)
            hand = v[:n] + ((g * w["w_hyp"]).sum(1) - v[:n] * w["hsum"])
            size = (np.abs(v[:n]) * (1 + np.abs(w["hsum"])) +
                    (np.abs(g) * np.abs(w["w_hyp"])).sum(1))
            assert (np.abs(hand - q) <= 2 * K * np.finfo(float).eps * size).all()
    got = [v.copy() for v in f]
    p = [a.ctypes.data_as(C.POINTER(C.c_double)) for a in got]
    s._ck(sunset_amd.lib().sv_filter_variables(s.h, *p))
    for a, v, q in zip(got[1:], f[1:], want[1:]):
        assert np.array_equal(a[:n], q) and np.array_equal(a[n:], v[n:])
    dev = (want[0] - 1.0) * w["vol"]
    ro = want[0] - dev.sum() / w["vol"].sum()
    bound = 4 * n * np.finfo(float).eps * np.abs(dev).sum() / w["vol"].sum() + 4e-16
    assert np.abs(got[0][:n] - ro).max() <= bound
    assert np.array_equal(got[0][n:], f[0][n:])
    s.close()
