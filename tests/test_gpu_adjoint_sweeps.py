"""The adjoint's halo-staged transposed gathers against its gathers from memory
("adj_lanes" 1), on node counts at the edges of their blocks and of the rule by
which the filter makes the mass sum itself (128 blocks), with wide and uneven
stencils and with polymer diffusion; and the reverse sweep from a tape that
the rollout wrote against one that computes the interval again.

Tolerance of the first: both add the same products, in another order; K links
change a sum by at most K roundings of its terms' sizes, which a step within the
stability limit weighs with O(10) at most: 4 stages * 6 steps * 10 * 100 *
1.1e-16 = 2.6e-12 of the largest value, 1e-11 allowed.  The second: bitwise."""
import dataclasses

import numpy as np
import pytest

from sunset_amd.nodes import jittered_lattice, perturbed_rest_ic

pytestmark = pytest.mark.gpu

KEYS = ("ro", "rou", "rov", "cxx", "cxy", "cyy")
PH = dict(Re=1.0, Wi=1.0, beta=0.5, eps=0.1, Ma=0.1, kol_amp=1.0, kol_k=4 * np.pi)


def _problem(nx, ny, order, uneven):
    ns = jittered_lattice(nx, ny, seed=nx, h_over_s={4: 1.8, 6: 2.4, 8: 2.7}[order],
                          box=(0.0, 1.0, 0.0, ny / nx))
    if uneven:                    # lists that are not symmetric
        f = 1.0 + 0.12 * np.sin(2 * np.pi * ns.x)
        ns = dataclasses.replace(ns, h=ns.h * f, h_small=ns.h_small * f * 0.97)
    ic = perturbed_rest_ic(ns, amp=0.05, seed=3)
    ic["cxx"] = 1.0 + 0.2 * np.sin(2 * np.pi * ns.x) ** 2
    ic["cxy"] = 0.1 * np.cos(2 * np.pi * ns.y)
    U = dict(ro=ic["ro"], rou=ic["ro"] * ic["u"], rov=ic["ro"] * ic["v"], cxx=ic["cxx"],
             cxy=ic["cxy"], cyy=ic["cyy"])
    return ns, U


@pytest.mark.parametrize("nx,ny,order,mdiff,uneven", [
    (17, 15, 6, 0.0, False),      # 255 nodes: one block, a slot short
    (16, 16, 4, 2e-3, False),     # exactly one block
    (33, 31, 4, 0.0, True),       # one ragged slice of the last block
    (40, 37, 8, 2e-3, True),      # wide stencils
    (181, 181, 4, 0.0, False),    # 128 blocks: the filter makes the mass sum
    (182, 181, 4, 0.0, False),    # 129: a kernel of its own does
])
def test_staged_gathers_match_memory_gathers(nx, ny, order, mdiff, uneven):
    import sunset_amd
    print(f"[adjoint sweeps] {nx}x{ny} order {order} Mdiff {mdiff} uneven {uneven}", flush=True)
    ns, U = _problem(nx, ny, order, uneven)
    dt = 0.02 / nx ** 2 * 16 if nx < 100 else 2e-6
    out = []
    for lanes in (1, 0):
        s = sunset_amd.Solver(morder=order, form="di").setup(ns)
        s.set_phys(**PH, Mdiff=mdiff)
        s.set_option("adj_lanes", lanes)
        s.set_state(U, dt=min(dt, 1e-5))
        s.adj_setup(4)
        L = s.rollout_forward(6)
        out.append((L, s.rollout_vjp(1.0), np.array(list(s.adj_param_grad().values()))))
        s.close()
    (La, ga, pa), (Lb, gb, pb) = out
    assert La == Lb
    for k in KEYS:
        assert np.isfinite(ga[k]).all(), k
        assert np.abs(ga[k] - gb[k]).max() <= 1e-11 * np.abs(ga[k]).max(), k
    assert np.abs(pa - pb).max() <= 1e-11 * np.abs(pa).max()


@pytest.mark.parametrize("steps,every", [(5, 5), (7, 3), (3, 8), (40, 36)])
def test_tape_of_the_rollout(steps, every):
    """The first reverse sweep reads the rollout's tape, the second (and one after
    new physics) computes the interval again; a rollout after one that nothing
    read writes none."""
    import sunset_amd
    ns, U = _problem(20, 19, 4, False)
    s = sunset_amd.Solver(morder=4, form="di").setup(ns)
    s.set_phys(**PH)
    s.set_state(U, dt=1e-5)
    s.adj_setup(every)
    L = s.rollout_forward(steps)
    first = s.rollout_vjp(1.0)
    p1 = s.adj_param_grad()
    again = s.rollout_vjp(1.0)
    p2 = s.adj_param_grad()
    grads = [again]
    for unread in (1, 2):
        for _ in range(unread):
            s.set_state(U, dt=1e-5)
            assert s.rollout_forward(steps) == L
        grads.append(s.rollout_vjp(1.0))
    s.set_state(U, dt=1e-5)
    s.rollout_forward(steps)
    s.set_phys(**PH)
    grads.append(s.rollout_vjp(1.0))
    for g in grads:
        for k in KEYS:
            assert np.array_equal(g[k], first[k]), k
    assert p1 == p2
    s.close()
