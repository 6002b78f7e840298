"""A node set that is refused leaves none: nothing runs on what was there before it,
and the next one is whole."""
import ctypes as C

import numpy as np
import pytest

from sunset_amd.nodes import jittered_lattice

pytestmark = pytest.mark.gpu


def test_refused_node_set_leaves_none():
    import sunset_amd
    print("[refused nodes]", flush=True)
    ns = jittered_lattice(20, 19, seed=20, h_over_s=1.8, box=(0.0, 1.0, 0.0, 0.95))
    s = sunset_amd.Solver(morder=4, form="lc").setup(ns)
    nt = np.full(ns.npfb, 7, np.int32)                    # no such node type
    p = [np.ascontiguousarray(a) for a in (ns.x, ns.y, ns.s, ns.h, ns.h_small)]
    D = C.POINTER(C.c_double)
    rc = sunset_amd.lib().sv_set_nodes(s.h, ns.npfb, *[a.ctypes.data_as(D) for a in p],
                                       nt.ctypes.data_as(C.POINTER(C.c_int32)))
    assert rc != 0
    with pytest.raises(sunset_amd.SunsetError, match="sv_set_nodes must come first"):
        s.find_neighbours(copy=False)
    with pytest.raises(sunset_amd.SunsetError, match="sv_find_neighbours must come first"):
        s.calc_weights()
    with pytest.raises(sunset_amd.SunsetError):
        s.laplacian(np.ones(s.np))
    t = sunset_amd.Solver(morder=4, form="lc").setup(ns)
    s.setup(ns)                                           # and the next one is whole
    phi = np.sin(np.arange(s.np))
    assert np.array_equal(s.laplacian(phi), t.laplacian(phi))
    s.close()
    t.close()
