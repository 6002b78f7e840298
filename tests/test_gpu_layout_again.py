"""What a context holds of its time-loop layout when the layout is made again:
captured steps, the transposed lists of the adjoint and boundary records do not
outlive it."""
import numpy as np
import pytest

from sunset_amd.nodes import jittered_lattice, perturbed_rest_ic, taylor_green_ic, wall_channel

pytestmark = pytest.mark.gpu

PH = dict(Re=1.0, Wi=1.0, beta=0.5, eps=0.1, Ma=0.1)
KEYS = ("ro", "rou", "rov", "cxx", "cxy", "cyy")


def _lattice(order=4):
    return jittered_lattice(20, 19, seed=20, h_over_s={4: 1.8, 6: 2.4}[order],
                            box=(0.0, 1.0, 0.0, 0.95))


def _again(s, order_map=None):
    """the lists and weights once more"""
    s.find_neighbours(copy=False)
    s.calc_weights(order_map)
    s.calc_sums()
    s.filter_coefficients()


def test_graphs_go_with_the_layout():
    import sunset_amd
    print("[layout again] graphs", flush=True)
    ns = _lattice()
    pair = []
    for _ in range(2):
        s = sunset_amd.Solver(morder=4, form="lc").setup(ns)
        s.set_phys(**PH)
        s.set_initial(taylor_green_ic(ns), dt=1e-6, itime=3)
        pair.append(s)
    s, t = pair
    s.run(4, graph=True)
    _again(s)
    E = sunset_amd.Ensemble([s])          # makes the member's layout again
    s.run(4, graph=True)
    assert s.timing("graph_steps") == 4
    t.run(4)
    E.run(4, graph=True)
    t.run(4)
    a, b, e = s.fields(), t.fields(), E.fields(0)
    for k in KEYS + ("dt", "time"):
        assert np.array_equal(a[k], b[k]) and np.array_equal(e[k], b[k]), k
    E.close()
    s.close()
    t.close()


def test_adjoint_of_new_weights():
    """order-4 weights on an order-6 context's lists after gradients with its own"""
    import sunset_amd
    print("[layout again] adjoint", flush=True)
    ns = _lattice(6)
    ic = perturbed_rest_ic(ns, amp=0.05, seed=3)
    U = dict(ro=ic["ro"], rou=ic["ro"] * ic["u"], rov=ic["ro"] * ic["v"],
             cxx=1.0 + 0.2 * np.sin(2 * np.pi * ns.x) ** 2, cxy=0.1 * np.cos(2 * np.pi * ns.y),
             cyy=np.ones(ns.npfb))
    four = np.full(ns.npfb, 4, np.int32)

    def gradient(s, setup):
        s.set_state(U, dt=1e-5)
        if setup:
            s.adj_setup(3)
        L = s.rollout_forward(5)
        return L, s.rollout_vjp(1.0), s.adj_param_grad()
    s = sunset_amd.Solver(morder=6, form="di").setup(ns)
    s.set_phys(**PH)
    first = gradient(s, True)
    _again(s)                             # the same weights: the same layout, made again
    same = gradient(s, False)
    _again(s, four)
    new = gradient(s, False)
    t = sunset_amd.Solver(morder=6, form="di").setup(ns, order_map=four)
    t.set_phys(**PH)
    want = gradient(t, True)
    for a, b in ((same, first), (new, want)):
        assert a[0] == b[0] and a[2] == b[2]
        for k in KEYS:
            assert np.isfinite(b[1][k]).all() and np.array_equal(a[1][k], b[1][k]), k
    assert new[0] != first[0]
    s.close()
    t.close()


def test_boundary_records_go_with_the_layout():
    """a state of boundary nodes is set again after their stencils"""
    import sunset_amd
    print("[layout again] boundary records", flush=True)
    ns = wall_channel(16, 16, order=4, seed=1)
    ic = perturbed_rest_ic(ns, amp=0.01, seed=3)
    s = sunset_amd.Solver(morder=4, form="lc").setup(ns)
    s.set_phys(**PH)
    s.set_initial(ic, dt=1e-7, itime=3)
    s.run(2)
    want = s.fields()
    s.find_neighbours(copy=False)
    s.calc_weights()
    s.calc_boundary_weights()
    s.calc_sums()
    s.filter_coefficients()
    with pytest.raises(sunset_amd.SunsetError, match="sv_set_initial, which must follow"):
        sunset_amd.Ensemble([s])
    with pytest.raises(sunset_amd.SunsetError, match="sv_set_initial must come first"):
        s.run(1)
    s.set_initial(ic, dt=1e-7, itime=3)
    s.run(2)
    got = s.fields()
    for k in KEYS:
        assert np.isfinite(want[k]).all() and np.array_equal(got[k], want[k]), k
    s.close()
