"""When a rollout writes the tape of its last checkpoint interval and when the
reverse sweep reads it ("rollout_tape"): as asked for, without memory taken by a
rollout that nothing differentiates, and never across new physics.  The gradient
from a tape is that of a reverse sweep which computes the interval again, bit for
bit (the same kernels write the same tape)."""
import numpy as np
import pytest

from sunset_amd.nodes import jittered_lattice, perturbed_rest_ic

pytestmark = pytest.mark.gpu

KEYS = ("ro", "rou", "rov", "cxx", "cxy", "cyy")
PH = dict(Re=1.0, Wi=1.0, beta=0.5, eps=0.1, Ma=0.1, kol_amp=1.0, kol_k=4 * np.pi)
NEW = dict(PH, Wi=0.6, eps=0.3)
DT = 1e-5


def _solver():
    import sunset_amd
    ns = jittered_lattice(20, 19, seed=20, h_over_s=1.8, box=(0.0, 1.0, 0.0, 0.95))
    ic = perturbed_rest_ic(ns, amp=0.05, seed=3)
    ic["cxx"] = 1.0 + 0.2 * np.sin(2 * np.pi * ns.x) ** 2
    ic["cxy"] = 0.1 * np.cos(2 * np.pi * ns.y)
    U = dict(ro=ic["ro"], rou=ic["ro"] * ic["u"], rov=ic["ro"] * ic["v"], cxx=ic["cxx"],
             cxy=ic["cxy"], cyy=ic["cyy"])
    s = sunset_amd.Solver(morder=4, form="di").setup(ns)
    s.set_phys(**PH)
    s.set_state(U, dt=DT)
    return s, U


def _stat(s):
    return tuple(int(s.timing(k)) for k in ("tape_steps", "tape_written", "vjp_recomputed"))


def _same(a, b):
    return all(np.array_equal(a[k], b[k]) for k in KEYS)


# last: steps of the last interval; held: steps of the longest
@pytest.mark.parametrize("steps,every,last,held", [(5, 5, 5, 5), (7, 3, 1, 3), (3, 8, 3, 3)])
@pytest.mark.parametrize("tape", [-1, 0, 1])
def test_when_a_tape_is_written(tape, steps, every, last, held):
    print(f"[tape] {tape} {steps}/{every}", flush=True)
    s, U = _solver()
    s.set_option("rollout_tape", tape)
    s.adj_setup(every)

    def forward():
        s.set_state(U, dt=DT)
        s.rollout_forward(steps)
        return _stat(s)[:2]

    def reverse():
        g = s.rollout_vjp(1.0)
        return g, _stat(s)[2]

    assert forward() == ((last, 1) if tape == 1 else (0, 0))   # no memory unless asked for
    g, again = reverse()
    assert again == (steps - last if tape == 1 else steps)
    g2, again = reverse()                      # the tape was used up
    assert again == steps and _same(g, g2)
    assert forward() == (held, int(tape != 0))
    g2, again = reverse()
    assert again == (steps if tape == 0 else steps - last) and _same(g, g2)
    assert forward() == (held, int(tape != 0))
    assert forward() == (held, int(tape == 1))  # the one before had no reverse sweep
    assert _stat(s)[0] == held
    s.close()


def test_new_physics_after_the_rollout():
    """the reverse sweep is that of the values in force when it runs"""
    out = {}
    for tape, ph in ((1, PH), (0, NEW), (1, NEW)):
        s, U = _solver()
        s.set_option("rollout_tape", tape)
        s.adj_setup(5)
        s.rollout_forward(5)
        s.set_phys(**ph)
        assert _stat(s)[1] == 0
        out[tape, ph["Wi"]] = s.rollout_vjp(1.0), s.adj_param_grad()
        assert _stat(s)[2] == 5
        s.close()
    (g, p), (g0, p0), (old, pold) = out[1, NEW["Wi"]], out[0, NEW["Wi"]], out[1, PH["Wi"]]
    assert _same(g, g0) and p == p0
    assert not _same(g, old) and p != pold


def test_autograd_asks_for_the_tape():
    """evaluations take no memory for one; a gradient reads the one of its own
    rollout, also between evaluations"""
    torch = pytest.importorskip("torch")
    from sunset_amd.autograd import rollout_loss
    s, U = _solver()
    U0 = torch.tensor(np.stack([U[k] for k in KEYS]))
    Wi = torch.tensor(1.0, dtype=torch.float64)

    def evaluate(u):
        return float(rollout_loss(s, u, 6, DT, checkpoint_every=4, Wi=Wi))

    L = evaluate(U0)
    with torch.no_grad():
        assert evaluate(U0.clone().requires_grad_(True)) == L
    assert _stat(s)[:2] == (0, 0)
    grads = []
    for _ in range(3):
        u = U0.clone().requires_grad_(True)
        w = Wi.clone().requires_grad_(True)
        loss = rollout_loss(s, u, 6, DT, checkpoint_every=4, Wi=w)
        assert _stat(s)[1] == 1
        loss.backward()
        assert _stat(s)[2] == 4              # the first interval; the last had its tape
        grads.append((u.grad, w.grad))
        assert evaluate(U0) == L and _stat(s)[1] == 0
    w = Wi.clone().requires_grad_(True)      # a gradient of a parameter alone
    rollout_loss(s, U0, 6, DT, checkpoint_every=4, Wi=w).backward()
    assert _stat(s)[2] == 4
    for gu, gw in grads:
        assert torch.equal(gu, grads[0][0]) and gw == grads[0][1] == w.grad
    s.close()
