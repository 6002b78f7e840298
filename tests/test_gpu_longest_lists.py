"""The longest neighbour lists: 1365 links are taken, up to the filter coefficients
(which stage whole lists in LDS), and one link more is refused by the search, so
that nothing after it meets a longer list."""
import dataclasses

import numpy as np
import pytest

import sunset_amd
from sunset_amd.nodes import jittered_lattice

LONGEST = 1365


def _nodes(kmax):
    """A periodic lattice whose longest list has kmax links (each node's own among
    them), and the lists' lengths."""
    ns = jittered_lattice(48, 47, seed=3, h_over_s=1.8)
    x = np.concatenate([ns.x + a for a in (-1, 0, 1) for _ in (-1, 0, 1)])
    y = np.concatenate([ns.y + b for _ in (-1, 0, 1) for b in (-1, 0, 1)])
    r = np.array([np.sort(np.hypot(x - ns.x[i], y - ns.y[i]))[kmax - 1:kmax + 1]
                  for i in range(ns.npfb)])
    lo, hi = r[:, 0].min(), r[:, 1].min()
    assert hi / lo - 1 > 1e-9                 # a radius between, beyond rounding
    h = np.full(ns.npfb, 0.25 * (lo + hi))
    return dataclasses.replace(ns, h=h, h_small=h.copy(), smax=6 * ns.smax)   # the search
    #                                           cells follow smax


def test_node_set_is_as_long_as_it_says():
    ns = _nodes(LONGEST)
    n = ns.npfb
    k = 0
    for i in range(n):
        dx = np.abs(ns.x - ns.x[i])[None, :] + np.array([[0.0], [-1.0], [1.0]])
        dy = np.abs(ns.y - ns.y[i])[None, :] + np.array([[0.0], [-1.0], [1.0]])
        k = max(k, int(((dx[:, None] ** 2 + dy[None] ** 2) <= (2 * ns.h[i]) ** 2).sum()))
    assert k == LONGEST


@pytest.mark.gpu
def test_longest_lists():
    print("[longest lists]", flush=True)
    s = sunset_amd.Solver(morder=4)
    s.set_nodes(_nodes(LONGEST))
    s.find_neighbours(copy=False)
    assert s.stencil_stats()["K_max"] == LONGEST
    s.calc_weights()
    s.calc_sums()
    b = s.weights(LONGEST)
    s.filter_coefficients()
    c = s.weights(LONGEST)
    s.close()
    eps = np.finfo(float).eps
    nz = b["w_hyp"] != 0
    assert nz.sum(1).max() == LONGEST - 1         # all but the node itself
    fac = np.where(nz, c["w_hyp"] / np.where(nz, b["w_hyp"], 1.0), np.nan)
    assert np.nanmax(np.nanmax(fac, 1) / np.nanmin(fac, 1) - 1.0) < 8 * eps   # one factor a row
    seq = np.cumsum(c["w_hyp"], axis=1)[:, -1]
    assert (np.abs(seq - c["hsum"]) <= LONGEST * eps * np.abs(c["w_hyp"]).sum(1)).all()


@pytest.mark.gpu
def test_longer_lists_are_refused():
    print("[longer lists]", flush=True)
    s = sunset_amd.Solver(morder=4)
    s.set_nodes(_nodes(LONGEST + 1))
    with pytest.raises(sunset_amd.SunsetError, match="1366 entries too long"):
        s.find_neighbours(copy=False)
    with pytest.raises(sunset_amd.SunsetError, match="sv_find_neighbours"):
        s.calc_weights()
    s.close()
