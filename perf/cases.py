"""The work that a user of this framework has it do, as measurable cases.

Each case is one pass through the public entry points (`sunset_amd.Solver`,
`Ensemble`, `autograd.rollout_loss`, the C ABI's device-pointer operators):

  march      a resident solver takes a state from device tensors, advances a
             number of RK3 steps and gives the registers back in device tensors
  channel    a wall-bounded channel advanced a number of steps, the fields
             copied to the host as an output interval does
  gradient   loss and gradients of a rollout through torch.autograd
  ensemble   several independent simulations advanced in one captured graph,
             the fields of every member read back
  operators  derivative operators and filter applied to device fields
  start      a new node set: lists, weights, sums, filter, loop layout, initial
             state, one step
  weights    lists, weights, sums and filter of a resident node set with an
             order map, the operators applied to one field
  adapt      the stencil adaptation of a new node set

Sizes are those of this repository's tests and benchmark (64^2, 128^2, 512^2,
1024^2 lattices, the cylinder channel at spacing 0.004..0.016, the log-uniform
ensemble) and odd, ragged ones between them.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch   # before the package: the library then shares torch's HIP runtime

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "sunset-viscoelastic_amd"))

import sunset_amd  # noqa: E402
from sunset_amd.autograd import rollout_loss  # noqa: E402
from sunset_amd import nodes  # noqa: E402

HOVS = {4: 1.8, 6: 2.4, 8: 2.7}
OP_GRAD, OP_LAP, OP_FILTER = 0, 1, 4
REG = ("ro", "rou", "rov", "pxx", "pxy", "pyy")
FLUID = dict(Re=1.0, Ma=0.1)


def listed():
    return [
        # the smallest runs: 4k nodes, order 4, direct form at the CFL-limited
        # dt; eight small launches a step, so latency is everything
        dict(name="march_di_64_o4", kind="march", nx=64, ny=64, order=4, form="di", steps=20,
             dt="cfl", Wi=1.0, beta=0.5, eps=0.0, Mdiff=0.0, kol=0.0, graph=True, bc="periodic"),
        # a small log-conformation run with odd sides and the default PID control
        dict(name="march_lc_127_o6", kind="march", nx=127, ny=131, order=6, form="lc", steps=10,
             dt="pid", Wi=2.0, beta=0.1, eps=0.25, Mdiff=0.0, kol=1.0, graph=False,
             bc="periodic"),
        # an ordinary direct-form run, order 8 (the widest stencils of the
        # time loop), with polymer diffusion, ragged sides
        dict(name="march_di_301_o8", kind="march", nx=301, ny=283, order=8, form="di", steps=10,
             dt="pid", Wi=1.0, beta=0.5, eps=0.1, Mdiff=1.0e-3, kol=0.0, graph=False,
             bc="periodic"),
        # an ordinary run between mirror (no-slip) edges
        dict(name="march_lc_450_o4", kind="march", nx=450, ny=450, order=4, form="lc", steps=10,
             dt="fixed", Wi=0.5, beta=0.5, eps=0.0, Mdiff=0.0, kol=0.0, graph=False,
             bc="noslip"),
        # the headline run: 1M nodes, order 6, log-conformation sPTT, forced
        dict(name="march_lc_1024_o6", kind="march", nx=1024, ny=1024, order=6, form="lc",
             steps=10, dt="pid", Wi=2.0, beta=0.1, eps=0.25, Mdiff=0.0, kol=1.0, graph=False,
             bc="periodic"),
        # boundary nodes with characteristic conditions, an output interval of
        # 20 steps with every field copied to the host
        dict(name="channel_lc_260_o6", kind="channel", nx=260, order=6, form="lc", walls=True,
             steps=20),
        # reverse mode: loss and gradients of a 20-step rollout (one
        # checkpoint interval) on the 128^2 lattice
        dict(name="gradient_di_128_o6", kind="gradient", nx=128, ny=128, order=6, steps=20,
             every=20),
        # independent simulations of log-uniform sizes, orders 4 and 6
        dict(name="ensemble_di_8", kind="ensemble", members=8, specs=7, form="di", steps=20),
        # the drop-in operators on device fields, an odd lattice
        dict(name="operators_511_o6", kind="operators", nx=511, ny=513, order=6, fields=3),
        # a new simulation from its node set to its first step
        dict(name="start_lc_512_o6", kind="start", nx=512, ny=512, order=6, form="lc",
             hs=2.4),
        # uneven stencils of two orders in one call: the cylinder channel
        dict(name="weights_cylinder_o84", kind="weights", smin=0.004, smax=0.016),
        # stencil adaptation of a new node set
        dict(name="adapt_96_o6", kind="adapt", nx=96, ny=96, order=6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["march"] * 4 + ["channel", "gradient", "ensemble", "operators", "start",
                                       "weights", "adapt"])
    order = rng.choice([4, 6, 6, 8])
    form = rng.choice(["lc", "di"])
    if kind == "march":
        nx = _log(rng, 48, 900)
        ny = max(48, min(900, int(nx * rng.uniform(0.6, 1.4))))
        return dict(kind=kind, nx=nx, ny=ny, order=order, form=form,
                    steps=rng.choice([5, 10, 15]), dt=rng.choice(["pid", "fixed", "cfl"]),
                    Wi=round(math.exp(rng.uniform(math.log(0.2), math.log(5.0))), 3),
                    beta=round(rng.uniform(0.1, 0.9), 3), eps=rng.choice([0.0, 0.1, 0.25]),
                    Mdiff=1.0e-3 if form == "di" and rng.random() < 0.4 else 0.0,
                    kol=rng.choice([0.0, 1.0]), graph=rng.random() < 0.5,
                    bc=rng.choice(["periodic", "noslip"]) if order == 4 else "periodic")
    if kind == "channel":
        return dict(kind=kind, nx=_log(rng, 48, 300), order=rng.choice([4, 6]), form=form,
                    walls=rng.random() < 0.6, steps=rng.choice([10, 20, 30]))
    if kind == "gradient":
        nx = _log(rng, 40, 224)
        return dict(kind=kind, nx=nx, ny=max(40, int(nx * rng.uniform(0.7, 1.2))),
                    order=rng.choice([4, 6]), steps=rng.choice([10, 20, 30]),
                    every=rng.choice([5, 10, 20]))
    if kind == "ensemble":
        return dict(kind=kind, members=rng.randint(2, 8), specs=rng.randint(100, 10 ** 6),
                    form=form, steps=rng.choice([10, 20]))
    if kind == "operators":
        nx = _log(rng, 48, 1000)
        return dict(kind=kind, nx=nx, ny=max(48, min(1000, int(nx * rng.uniform(0.6, 1.4)))),
                    order=order, fields=rng.randint(1, 4))
    if kind == "start":
        nx = _log(rng, 48, 600)
        return dict(kind=kind, nx=nx, ny=max(48, int(nx * rng.uniform(0.7, 1.1))), order=order,
                    form=form, hs=round(HOVS[order] * rng.choice([1.0, 1.0, 0.95]), 4))
    if kind == "weights":
        smin = round(math.exp(rng.uniform(math.log(0.004), math.log(0.02))), 5)
        return dict(kind=kind, smin=smin, smax=round(smin * rng.uniform(2.0, 4.0), 5))
    return dict(kind="adapt", nx=_log(rng, 32, 128), ny=_log(rng, 32, 110),
                order=rng.choice([4, 6]))


# ---- inputs -----------------------------------------------------------------

def _lattice(case, seed, hs=None):
    """A jittered lattice on [0,1] x [0, ny/nx] (spacing 1/nx), lists of h = hovs*s."""
    nx, ny, order = case["nx"], case["ny"], case["order"]
    s = 1.0 / nx
    rng = np.random.default_rng([seed, 1])
    i, j = (a.ravel() for a in np.meshgrid(np.arange(nx), np.arange(ny), indexing="ij"))
    x = (i + 0.5 + rng.uniform(-0.3, 0.3, i.size)) * s
    y = (j + 0.5 + rng.uniform(-0.3, 0.3, i.size)) * s
    n = x.size
    bc = (1, 1, 3, 3) if case.get("bc") == "noslip" else (1, 1, 1, 1)
    return nodes.NodeSet(x=x, y=y, s=np.full(n, s), h=np.full(n, HOVS[order] * s),
                         h_small=np.full(n, (HOVS[order] if hs is None else hs) * s),
                         node_type=np.full(n, 999, dtype=np.int32), xmin=0.0, xmax=1.0, ymin=0.0,
                         ymax=ny * s, bc=bc, smax=s)


def _waves(rng, x, y, Ly, modes=4, kmax=3):
    """A smooth random field of unit size, periodic on [0,1] x [0,Ly]."""
    f = np.zeros_like(x)
    for _ in range(modes):
        kx, ky = int(rng.integers(-kmax, kmax + 1)), int(rng.integers(1, kmax + 1))
        f += rng.uniform(0.3, 1.0) * np.cos(2 * np.pi * (kx * x + ky * y / Ly)
                                            + rng.uniform(0, 2 * np.pi))
    return f / math.sqrt(0.3 * modes)


def _flow(ns, seed, amp=0.5, still=None):
    """A developed viscoelastic flow: density near 1, velocities of order one,
    a positive definite conformation tensor exp(S) of moderate stretch.  still
    (values 0..1 per node): damps velocity and stretch towards walls."""
    rng = np.random.default_rng([seed, 2])
    Ly = ns.ymax - ns.ymin
    w = [_waves(rng, ns.x, ns.y, Ly) for _ in range(6)]
    d = 1.0 if still is None else still
    ro = 1.0 + 0.002 * w[0] * d
    u, v = amp * w[1] * d, amp * w[2] * d
    a, b, c = (0.3 + 0.15 * w[3]) * d + 0.02, (0.12 * w[4]) * d, (-0.1 + 0.1 * w[5]) * d
    cxx, cxy, cyy = _sym(np, a, b, c, np.exp)
    return dict(ro=ro, u=u, v=v, cxx=cxx, cxy=cxy, cyy=cyy)


def _sym(xp, a, b, c, f):
    """f of the symmetric 2x2 matrices [[a, b], [b, c]], by their principal axes."""
    th = 0.5 * xp.arctan2(2.0 * b, a - c)
    co, si = xp.cos(th), xp.sin(th)
    m, r = 0.5 * (a + c), xp.sqrt(0.25 * (a - c) ** 2 + b * b)
    f1, f2 = f(m + r), f(m - r)
    return f1 * co * co + f2 * si * si, (f1 - f2) * co * si, f1 * si * si + f2 * co * co


def _registers(ic, form):
    ro = ic["ro"]
    f = (_sym(np, ic["cxx"], ic["cxy"], ic["cyy"], np.log) if form == "lc"
         else (ic["cxx"], ic["cxy"], ic["cyy"]))
    return np.stack([ro, ro * ic["u"], ro * ic["v"], *f])


def _dt(case, s):
    """A step well inside the acoustic and viscous limits of spacing s."""
    return 0.25 * min(s / 11.0, 2.0 / 3.0 * s * s)


def _phys(case):
    return dict(FLUID, Wi=case["Wi"], beta=case["beta"], eps=case["eps"], Mdiff=case["Mdiff"],
                kol_amp=case["kol"], kol_k=4 * math.pi)


GRAD_PHYS = dict(FLUID, Wi=1.0, beta=0.5, eps=0.1, kol_amp=1.0, kol_k=4 * math.pi)
START_PHYS = dict(FLUID, Wi=2.0, beta=0.1, eps=0.25)
MODES = {"pid": 0, "fixed": 1, "cfl": 2}


def _state_of(case, seed):
    ns = _lattice(case, seed)
    still = None
    if case.get("bc") == "noslip":
        still = np.sin(np.pi * (ns.y - ns.ymin) / (ns.ymax - ns.ymin))
    return ns, _flow(ns, seed, still=still)


def _channel_of(case, seed):
    n = case["nx"]
    make = nodes.wall_channel if case["walls"] else nodes.inflow_outflow_channel
    ns = make(n, n, order=case["order"], seed=seed)
    if case["walls"]:
        prof = 4.0 * ns.y * (1.0 - ns.y)
        ic = _flow(ns, seed, amp=0.1, still=prof)
        ic["u"] = ic["u"] + 0.5 * prof
    else:
        ic = _flow(ns, seed, amp=0.05, still=np.sin(np.pi * ns.x) ** 2)
        ic["u"] = ic["u"] + 0.5
    return ns, ic


def _members_of(case, seed):
    out = []
    for k, (side, order, Wi, beta) in enumerate(nodes.ensemble_specs(case["members"],
                                                                     case["specs"])):
        c = dict(nx=side, ny=side, order=order)
        ns = _lattice(c, [seed, k])
        out.append((c, ns, _flow(ns, seed + 7 * k), Wi, beta))
    return out


def _field_of(ns, seed, k=0):
    rng = np.random.default_rng([seed, 3, k])
    return 1.0 + 0.5 * _waves(rng, ns.x, ns.y, ns.ymax - ns.ymin)


def _cylinder_of(case, seed):
    """The channel's node set (its count is the generator's), the fluid nodes
    moved a little further by the seed; those on the cylinder stay."""
    ns, om = nodes.cylinder_channel(smin=case["smin"], smax=case["smax"])
    rng = np.random.default_rng([seed, 1])
    free = np.hypot(ns.x - 2.0, ns.y - 1.0) > 0.5 + 1e-9
    ns.x = ns.x + np.where(free, rng.uniform(-0.05, 0.05, ns.npfb) * ns.s, 0.0)
    ns.y = ns.y + np.where(free, rng.uniform(-0.05, 0.05, ns.npfb) * ns.s, 0.0)
    return ns, om


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda:0")


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case, kind=kind)
    if kind == "march":
        ns, ic = _state_of(case, seed)
        s = sunset_amd.Solver(morder=case["order"], form=case["form"]).setup(ns)
        s.set_phys(**_phys(case))
        s.set_initial(ic, dt=_dt(case, ns.smax), itime=10, dt_mode=case["dt"])
        U0 = _dev(_registers(ic, case["form"]))
        st.update(s=s, U0=U0, U=torch.empty_like(U0), dt=_dt(case, ns.smax))
    elif kind == "channel":
        ns, ic = _channel_of(case, seed)
        s = sunset_amd.Solver(morder=case["order"], form=case["form"]).setup(ns)
        s.set_phys(**START_PHYS, drive=(2.0 if case["walls"] else 0.0, 0.0, 0.0))
        s.set_initial(ic, dt=0.2 * _dt(case, ns.smax), itime=10)
        F = s.fields()
        keys = REG if case["form"] == "lc" else REG[:3] + ("cxx", "cxy", "cyy")
        st.update(s=s, U0=_dev(np.stack([F[k] for k in keys])), dt=0.2 * _dt(case, ns.smax))
    elif kind == "gradient":
        ns, ic = _state_of(case, seed)
        s = sunset_amd.Solver(morder=case["order"], form="di").setup(ns)
        s.set_phys(**GRAD_PHYS)
        st.update(s=s, U0=_dev(_registers(ic, "di")), dt=_dt(case, ns.smax))
    elif kind == "ensemble":
        ms = []
        for c, ns, ic, Wi, beta in _members_of(case, seed):
            s = sunset_amd.Solver(morder=c["order"], form=case["form"]).setup(ns)
            s.set_phys(**FLUID, Wi=Wi, beta=beta, kol_amp=1.0, kol_k=4 * math.pi)
            s.set_initial(ic, dt=_dt(c, ns.smax), itime=10)
            ms.append(s)
        st.update(E=sunset_amd.Ensemble(ms), n=len(ms))
    elif kind == "operators":
        ns = _lattice(case, seed)
        s = sunset_amd.Solver(morder=case["order"], form="lc").setup(ns)
        f = [_dev(_field_of(ns, seed, k)) for k in range(case["fields"])]
        n = ns.npfb
        st.update(s=s, f=f, g=[f[0].new_empty(2 * n) for _ in f], l=[f[0].new_empty(n) for _ in f],
                  h=[f[0].new_empty(n) for _ in f])
    elif kind == "start":
        ns = _lattice(case, seed, hs=case["hs"])
        st.update(ns=ns, ic=_flow(ns, seed), U=_dev(np.zeros((6, ns.npfb))),
                  s=sunset_amd.Solver(morder=case["order"], form=case["form"]))
    elif kind == "weights":
        ns, om = _cylinder_of(case, seed)
        s = sunset_amd.Solver(morder=8, form="lc")
        s.set_nodes(ns)
        f = _dev(_field_of(ns, seed))
        st.update(s=s, om=om, f=[f], g=[f.new_empty(2 * ns.npfb)], l=[f.new_empty(ns.npfb)],
                  h=[f.new_empty(ns.npfb)])
    elif kind == "adapt":
        st.update(ns=_lattice(case, seed),
                  s=sunset_amd.Solver(morder=case["order"], form="lc"))
    return st


# ---- one pass ---------------------------------------------------------------

def _ck(s, rc):
    if rc != 0:
        raise sunset_amd.SunsetError(sunset_amd.lib().sv_last_error(s.h).decode())


def _rows(U):
    return [U[q].data_ptr() for q in range(6)]


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _load(st, dt_mode):
    """The registers and the control state of a restart."""
    s, tol = st["s"], 1.0e-5
    s.set_state_device(_rows(st["U0"]), _stream())
    _ck(s, sunset_amd.lib().sv_set_control(s.h, st["dt"], 0.0, 10, tol, tol, tol, MODES[dt_mode]))


def _apply(st):
    """Gradient, Laplacian and filter of the fields, on torch's stream."""
    s, L, stream = st["s"], sunset_amd.lib(), ctypes.c_void_p(_stream() or None)
    nf = len(st["f"])
    arr = ctypes.c_void_p * nf
    src = arr(*[t.data_ptr() for t in st["f"]])
    for op, key in ((OP_GRAD, "g"), (OP_LAP, "l"), (OP_FILTER, "h")):
        _ck(s, L.sv_apply_dev(s.h, op, nf, src, arr(*[t.data_ptr() for t in st[key]]), stream))
    return dict(grad=st["g"], lap=st["l"], filt=st["h"])


def run(st):
    case, kind = st["case"], st["kind"]
    if kind == "march":
        _load(st, case["dt"])
        st["s"].run(case["steps"], graph=case["graph"])
        st["s"].get_state_device(_rows(st["U"]), _stream())
        return st["U"]
    if kind == "channel":
        _load(st, "pid")
        st["s"].run(case["steps"])
        F = st["s"].fields()
        return {k: F[k] for k in ("ro", "rou", "rov", "u", "v", "cxx", "cxy", "cyy", "dt")}
    if kind == "gradient":
        U = st["U0"].clone().requires_grad_(True)
        Wi, beta = (torch.tensor(v, dtype=torch.float64, requires_grad=True) for v in (1.0, 0.5))
        loss = rollout_loss(st["s"], U, case["steps"], st["dt"], checkpoint_every=case["every"],
                            Wi=Wi, beta=beta)
        loss.backward()
        return dict(loss=loss.detach(), U=U.grad, Wi=Wi.grad, beta=beta.grad)
    if kind == "ensemble":
        st["E"].run(case["steps"], graph=True)
        out = []
        for m in range(st["n"]):
            F = st["E"].fields(m)
            out.append(np.stack([F[k] for k in ("ro", "rou", "rov", "cxx", "cxy", "cyy")]))
        return out
    if kind == "operators":
        return _apply(st)
    if kind == "start":
        s = st["s"].setup(st["ns"])
        s.set_phys(**START_PHYS)
        s.set_initial(st["ic"], dt=_dt(case, st["ns"].smax), itime=10, dt_mode="fixed")
        s.run(1)
        s.get_state_device(_rows(st["U"]), _stream())
        return st["U"]
    if kind == "weights":
        s = st["s"]
        s.find_neighbours(copy=False)
        s.calc_weights(st["om"])
        s.calc_sums()
        s.filter_coefficients()
        return _apply(st)
    s = st["s"].set_nodes(st["ns"])
    s.find_neighbours(copy=False)
    h, hs, red = s.adapt_stencils()
    return dict(h=h, h_small=hs, reductions=red)


# ---- what a pass cannot do without -------------------------------------------

def _links(order, n):
    """Links of n lattice nodes: the lattice points in a disc of 2 hovs s."""
    return n * math.pi * (2.0 * HOVS[order]) ** 2


def _march_work(order, form, n, steps):
    """Each sweep (four stages, the filter) reads its weights and link targets
    once -- three or one FP64 weights and two bytes a link -- and its fields
    once and writes its results once; a sum is a multiply-add."""
    K, lc = _links(order, n), form == "lc"
    gather, state = (80 if lc else 48), 48
    stage = 26 * K + n * (2 * gather + 4 * state + 24)
    filt = 10 * K + n * (2 * state + 24)
    return dict(bytes=steps * (4 * stage + filt),
                flops=steps * K * (4 * 2 * (18 if lc else 14) + 12))


def _solve_work(order, n):
    """Assembly, elimination of an N x N system and evaluation of the weights."""
    N = (order * order + 3 * order) // 2
    K = _links(order, n)
    return dict(bytes=K * (4 + 16 + 32), flops=2 * K * N * N + n * 2.0 * N ** 3 / 3
                + 8 * n * N * N + 8 * K * N)


def work(case):
    kind = case["kind"]
    if kind == "march":
        return _march_work(case["order"], case["form"], case["nx"] * case["ny"], case["steps"])
    if kind == "channel":
        n = case["nx"] ** 2
        w = _march_work(case["order"], case["form"], n, case["steps"])
        return dict(bytes=w["bytes"] + 8 * 8 * n, flops=w["flops"])
    if kind == "gradient":
        # the forward steps, their recomputation and the transposed sweeps
        w = _march_work(case["order"], "di", case["nx"] * case["ny"], case["steps"])
        return dict(bytes=3 * w["bytes"], flops=3 * w["flops"])
    if kind == "ensemble":
        b = f = 0
        for side, order, _, _ in nodes.ensemble_specs(case["members"], case["specs"]):
            w = _march_work(order, case["form"], side * side, case["steps"])
            b, f = b + w["bytes"] + 48 * side * side, f + w["flops"]
        return dict(bytes=b, flops=f)
    if kind == "operators":
        n = case["nx"] * case["ny"]
        K = _links(case["order"], n)
        # targets and the four weights of a link once for all fields
        return dict(bytes=K * (4 + 32) + case["fields"] * n * 8 * 5,
                    flops=case["fields"] * K * 8)
    if kind == "start":
        n = case["nx"] * case["ny"]
        a, b = _solve_work(case["order"], n), _march_work(case["order"], case["form"], n, 1)
        return dict(bytes=a["bytes"] + b["bytes"], flops=a["flops"] + b["flops"])
    if kind == "weights":
        # nodes of the channel [0,8] x [0,2] at its mean spacing
        n = 16.0 / (0.8 * case["smax"] + 0.1 * case["smin"]) ** 2 * 1.2
        a = _solve_work(8, n)
        return dict(bytes=a["bytes"] + _links(8, n) * 36, flops=a["flops"] + _links(8, n) * 8)
    # about ten trial radii a node, each a moment matrix and its decomposition
    n = case["nx"] * case["ny"]
    N = (case["order"] ** 2 + 3 * case["order"]) // 2
    return dict(bytes=n * 48 + _links(case["order"], n) * 20,
                flops=10.0 * (2 * _links(case["order"], n) * N * N + n * 15.0 * N ** 3))


# ---- the same results in plain torch, 64 bits ---------------------------------

_CHUNK = 1 << 15


class _Stencils:
    """Lists, LABFM weights and filter of a node set without boundary nodes
    (periodic or open edges), as padded [n, K] arrays."""

    def __init__(self, ns, order, om=None):
        dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        t = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64, device=dev)  # noqa: E731
        self.x, self.y, self.h, self.hs, self.s = (t(a) for a in (ns.x, ns.y, ns.h, ns.h_small,
                                                                  ns.s))
        self.per = (ns.bc[0] == 1, ns.bc[2] == 1)
        self.box = (ns.xmin, ns.xmax - ns.xmin, ns.ymin, ns.ymax - ns.ymin)
        n = self.x.numel()
        self._cells()
        om = np.full(n, order) if om is None else np.asarray(om)
        K = int(self.count.max())
        z = lambda: torch.zeros(n, K, dtype=torch.float64, device=dev)  # noqa: E731
        self.col = torch.zeros(n, K, dtype=torch.int64, device=dev)
        self.wx, self.wy, self.wl, self.wh = z(), z(), z(), z()
        self.vol = torch.zeros(n, dtype=torch.float64, device=dev)
        for o in sorted(set(int(v) for v in np.unique(om))):
            ids = torch.as_tensor(np.nonzero(om == o)[0], device=dev)
            for a in range(0, ids.numel(), _CHUNK // 2):
                self._solve(ids[a:a + _CHUNK // 2], o, K)

    def _cells(self):
        x0, Lx, y0, Ly = self.box
        R = 2.0 * float(self.h.max())
        ncx, ncy = max(1, int(Lx / R)), max(1, int(Ly / R))
        cx = ((self.x - x0) / Lx * ncx).long().clamp(0, ncx - 1)
        cy = ((self.y - y0) / Ly * ncy).long().clamp(0, ncy - 1)
        c = cy * ncx + cx
        o = torch.argsort(c, stable=True)
        cnt = torch.bincount(c, minlength=ncx * ncy)
        first = torch.cumsum(cnt, 0) - cnt
        M = int(cnt.max())
        tab = torch.full((ncx * ncy + 1, M), -1, dtype=torch.int64, device=c.device)
        tab[c[o], torch.arange(c.numel(), device=c.device) - first[c[o]]] = o
        self.tab, self.cx, self.cy, self.ncx, self.ncy = tab, cx, cy, ncx, ncy
        self.count = torch.zeros_like(c)
        step = max(256, (1 << 26) // (9 * M))
        for a in range(0, c.numel(), step):
            ids = torch.arange(a, min(a + step, c.numel()), device=c.device)
            self.count[ids] = self._near(ids)[1].sum(1)

    def _near(self, ids):
        cand = []
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                qx, qy = self.cx[ids] + dx, self.cy[ids] + dy
                ok = torch.ones_like(qx, dtype=torch.bool)
                if self.per[0]:
                    qx = qx % self.ncx
                else:
                    ok &= (qx >= 0) & (qx < self.ncx)
                if self.per[1]:
                    qy = qy % self.ncy
                else:
                    ok &= (qy >= 0) & (qy < self.ncy)
                cand.append(self.tab[torch.where(ok, qy * self.ncx + qx, self.ncx * self.ncy)])
        j = torch.cat(cand, 1)
        dx, dy = self._d(ids, j.clamp(min=0))
        return j, (j >= 0) & (dx * dx + dy * dy <= (2.0 * self.h[ids, None]) ** 2)

    def _d(self, ids, j):
        dx, dy = self.x[j] - self.x[ids, None], self.y[j] - self.y[ids, None]
        if self.per[0]:
            dx = dx - self.box[1] * torch.round(dx / self.box[1])
        if self.per[1]:
            dy = dy - self.box[3] * torch.round(dy / self.box[3])
        return dx, dy

    @staticmethod
    def _powers(order, x, y):
        """Taylor monomials and Hermite products (probabilists'), by degree."""
        hx, hy, px, py = [x * 0 + 1, x], [y * 0 + 1, y], [x * 0 + 1, x], [y * 0 + 1, y]
        for k in range(1, order):
            hx.append(x * hx[k] - k * hx[k - 1])
            hy.append(y * hy[k] - k * hy[k - 1])
            px.append(px[k] * x / (k + 1))
            py.append(py[k] * y / (k + 1))
        mono = [px[d - b] * py[b] for d in range(1, order + 1) for b in range(d + 1)]
        herm = [hx[d - b] * hy[b] for d in range(1, order + 1) for b in range(d + 1)]
        return torch.stack(mono, -1), torch.stack(herm, -1)

    def _system(self, order, dx, dy, hh, inside):
        x, y = dx / hh, dy / hh
        q = torch.sqrt(x * x + y * y)
        w = torch.where((q <= 2.0) & (q > 0.0) & inside, (2 * q + 1) * (1 - 0.5 * q) ** 4, 0.0)
        mono, g = self._powers(order, x, y)
        g = g * w[..., None]
        used = torch.where(inside[..., None], mono, 0.0)
        return torch.matmul(used.transpose(1, 2).contiguous(), g), g

    def _solve(self, ids, order, K):
        pad = (1 << 27) // (9 * self.tab.shape[1])
        for a in range(0, ids.numel(), max(64, min(pad, _CHUNK // 4))):
            self._solve_some(ids[a:a + max(64, min(pad, _CHUNK // 4))], order, K)

    def _solve_some(self, ids, order, K):
        j, m = self._near(ids)
        at = torch.argsort((~m).to(torch.int8), dim=1, stable=True)[:, :K]
        j, m = torch.gather(j, 1, at), torch.gather(m, 1, at)
        if j.shape[1] < K:
            return self._solve_some(ids, order, j.shape[1])
        j = torch.where(m, j, ids[:, None])
        self.col[ids, :K] = j
        dx, dy = self._d(ids, j)
        r2 = dx * dx + dy * dy
        h, hs = self.h[ids, None], self.hs[ids, None]
        N = (order * order + 3 * order) // 2
        A, g = self._system(order, dx, dy, hs, m & (r2 <= (2 * hs) ** 2))
        b = A.new_zeros(ids.numel(), N, 3)
        b[:, 0, 0] = 1.0
        b[:, 1, 1] = 1.0
        b[:, 2, 2] = b[:, 4, 2] = 1.0
        w = torch.matmul(g, torch.linalg.solve(A, b))
        self.wx[ids, :K], self.wy[ids, :K] = w[..., 0] / hs, w[..., 1] / hs
        self.wl[ids, :K] = w[..., 2] / (hs * hs)
        # the highest even derivative (d/dx^2 + d/dy^2)^(order/2) for the filter
        A, g = self._system(order, dx, dy, h, m)
        p = order // 2
        b = A.new_zeros(ids.numel(), N, 1)
        for k in range(p + 1):
            b[:, N - (order + 1) + 2 * k, 0] = (-1.0) ** (p + 1) * math.comb(p, k)
        wh = torch.matmul(g, torch.linalg.solve(A, b))[..., 0]
        cnt = m.sum(1, keepdim=True).double()
        kk = (2.0 / 3.0) * math.pi / (2.0 * h * torch.sqrt(math.pi / cnt))
        amp = ((1.0 - torch.cos(kk * dx) * torch.cos(kk * dy)) * wh).sum(1, keepdim=True)
        self.wh[ids, :K] = wh * (2.0 / 3.0) / amp
        e = torch.where(m, torch.exp(-9.0 * r2 / (h * h)) * (9.0 / math.pi) / (h * h), 0.0)
        self.vol[ids] = 1.0 / e.sum(1)

    def sums(self, weights, F):
        """sum_j w_ij (F_j - F_i) for F [n, f] and each of the weights."""
        return _Sums.apply(F, self.col, *weights)

    def grads(self, F):
        return self.sums((self.wx, self.wy, self.wl), F)

    def filtered(self, F):
        return F + self.sums((self.wh,), F)[0]


class _Sums(torch.autograd.Function):
    @staticmethod
    def forward(ctx, F, col, *ws):
        ctx.save_for_backward(col, *ws)
        out = [torch.empty_like(F) for _ in ws]
        for a in range(0, F.shape[0], _CHUNK):
            b = slice(a, a + _CHUNK)
            D = F[col[b]] - F[b, None]
            for o, w in zip(out, ws):
                o[b] = (w[b, :, None] * D).sum(1)
        return tuple(out)

    @staticmethod
    def backward(ctx, *gs):
        col, *ws = ctx.saved_tensors
        G = torch.zeros_like(gs[0])
        for a in range(0, G.shape[0], _CHUNK):
            b = slice(a, a + _CHUNK)
            D = sum(w[b, :, None] * g[b, None] for g, w in zip(gs, ws))
            G.index_add_(0, col[b].reshape(-1), D.reshape(-1, D.shape[-1]))
            G[b] -= D.sum(1)
        return (G, None) + (None,) * len(ws)


_A = (11847461282814.0 / 36547543011857.0, 3943225443063.0 / 7078155732230.0,
      -346793006927.0 / 4029903576067.0)
_B = (1017324711453.0 / 9774461848756.0, 8237718856693.0 / 13685301971492.0,
      57731312506979.0 / 19404895981398.0, -101169746363290.0 / 37734290219643.0)
_BH = (15763415370699.0 / 46270243929542.0, 514528521746.0 / 5659431552419.0,
       27030193851939.0 / 9429696342944.0, -69544964788955.0 / 30262026368149.0)


class _Model:
    """The Oldroyd-B / sPTT equations on the stencils, RK3(2)4[2R+]C steps."""

    def __init__(self, S, form, Re=1.0, Wi=1.0, beta=0.5, eps=0.0, Ma=0.1, Mdiff=0.0,
                 kol_amp=0.0, kol_k=0.0):
        self.S, self.lc, self.eps, self.Md, self.lam = S, form == "lc", eps, Mdiff, Wi
        self.visc, self.csq = 1.0 / Re, 1.0 / Ma ** 2
        self.sol, self.pol = beta / Re, (1.0 - beta) / Re / Wi
        self.fx = kol_amp * torch.sin(kol_k * S.y)

    def rhs(self, U):
        ro, u, v = U[:, 0], U[:, 1] / U[:, 0], U[:, 2] / U[:, 0]
        if self.lc:
            p = U[:, 3:6].unbind(1)
            c = _sym(torch, *p, torch.exp)
            F = torch.stack([ro, u, v, *c, *p], 1)
        else:
            c = U[:, 3:6].unbind(1)
            F = torch.stack([ro, u, v, *c], 1)
        X, Y, L = self.S.grads(F)
        ux, uy, vx, vy = X[:, 1], Y[:, 1], X[:, 2], Y[:, 2]
        r_ro = -(u * X[:, 0] + v * Y[:, 0]) - ro * (ux + vy)
        r_u = (u * r_ro - ro * (u * ux + v * uy) - self.csq * X[:, 0] + self.fx
               + self.sol * L[:, 1] + self.pol * (X[:, 3] + Y[:, 4]))
        r_v = (v * r_ro - ro * (u * vx + v * vy) - self.csq * Y[:, 0]
               + self.sol * L[:, 2] + self.pol * (X[:, 4] + Y[:, 5]))
        if self.lc:
            r = self._logconf(u, v, ux, uy, vx, vy, p, X[:, 6:9], Y[:, 6:9])
        else:
            f = (1.0 - 2.0 * self.eps + self.eps * (c[0] + c[2] + 1.0)) / self.lam
            adv = [-(u * X[:, k] + v * Y[:, k]) + self.Md * L[:, k] for k in (3, 4, 5)]
            r = (adv[0] + 2 * (ux * c[0] + uy * c[1]) - f * (c[0] - 1.0),
                 adv[1] + ux * c[1] + uy * c[2] + vx * c[0] + vy * c[1] - f * c[1],
                 adv[2] + 2 * (vx * c[1] + vy * c[2]) - f * (c[2] - 1.0))
        return torch.stack([r_ro, r_u, r_v, *r], 1)

    def _logconf(self, u, v, ux, uy, vx, vy, p, X, Y):
        th = 0.5 * torch.arctan2(2 * p[1], p[0] - p[2])
        co, si = torch.cos(th), torch.sin(th)
        m, r = 0.5 * (p[0] + p[2]), torch.sqrt(0.25 * (p[0] - p[2]) ** 2 + p[1] ** 2)
        a1, a2 = torch.exp(m + r), torch.exp(m - r)
        # the velocity gradient in the principal axes
        m11 = co * co * ux + co * si * (uy + vx) + si * si * vy
        m22 = si * si * ux - co * si * (uy + vx) + co * co * vy
        m12 = co * (co * uy + si * vy) - si * (co * ux + si * vx)
        m21 = co * (co * vx - si * ux) + si * (co * vy - si * uy)
        # rotation times the eigenvalue difference; its limit at a1 = a2
        k = torch.where(r > 1e-9, 2 * r / (a2 - a1), -1.0 / a1)
        off = -k * (a2 * m12 + a1 * m21)
        fr = 1.0 - 2.0 * self.eps + self.eps * (a1 + a2)
        d1 = 2 * m11 + (fr / a1 - fr) / self.lam
        d2 = 2 * m22 + (fr / a2 - fr) / self.lam
        adv = [-(u * X[:, q] + v * Y[:, q]) for q in range(3)]
        return (adv[0] + d1 * co * co + d2 * si * si - 2 * co * si * off,
                adv[1] + (d1 - d2) * co * si + (co * co - si * si) * off,
                adv[2] + d1 * si * si + d2 * co * co + 2 * co * si * off)

    def limits(self, U):
        sp = torch.sqrt((U[:, 1] / U[:, 0]) ** 2 + (U[:, 2] / U[:, 0]) ** 2)
        s = self.S.s
        return min(float((s / (sp + math.sqrt(self.csq))).min()),
                   2.0 / 3.0 * float((s * s * U[:, 0]).min()) / self.visc)

    def step(self, U, dt):
        r, W, e = U, U, 0.0
        for k in range(4):
            R = dt * self.rhs(W)
            e = e + (_B[k] - _BH[k]) * R
            if k < 3:
                W = r + _A[k] * R
            r = r + _B[k] * R
        U = self.S.filtered(r)
        dro = ((U[:, 0] - 1.0) * self.S.vol).sum() / self.S.vol.sum()
        U = torch.cat([U[:, :1] - dro, U[:, 1:]], 1)
        return U, e

    def march(self, U, steps, dt, mode):
        em = [1e-5] * 3   # newest first
        for _ in range(steps):
            if mode != "fixed":
                top = self.limits(U)
                if mode == "cfl":
                    dt = top
                else:
                    f = 0.9 * ((1e-5 / em[0]) ** 0.245 * (em[1] / 1e-5) ** 0.17
                               * (1e-5 / em[2]) ** 0.05)
                    dt = min(dt * min(1.02, max(0.5, f)), top)
            U, e = self.step(U, dt)
            em = [max(float(e.abs().max()), 1e-16), em[0], em[1]] if mode == "pid" else em
        return U


def exact(case, seed):
    kind = case["kind"]
    if kind in ("channel", "adapt") or case.get("bc") == "noslip":
        # characteristic boundary conditions and one-sided operators; mirrored
        # edges; decisions of the adaptation, which have no value of their own
        return None
    if kind in ("march", "start"):
        ns = _lattice(case, seed, hs=case.get("hs"))
        M = _Model(_Stencils(ns, case["order"]), case["form"],
                   **(_phys(case) if kind == "march" else START_PHYS))
        U = _dev(_registers(_flow(ns, seed), case["form"])).T.contiguous()
        return M.march(U, case.get("steps", 1), _dt(case, ns.smax),
                       case.get("dt", "fixed")).T.contiguous()
    if kind == "ensemble":
        out = []
        for c, ns, ic, Wi, beta in _members_of(case, seed):
            M = _Model(_Stencils(ns, c["order"]), case["form"], **FLUID, Wi=Wi, beta=beta,
                       kol_amp=1.0, kol_k=4 * math.pi)
            U = M.march(_dev(_registers(ic, case["form"])).T.contiguous(), case["steps"],
                        _dt(c, ns.smax), "pid").T
            if case["form"] == "lc":
                U = torch.cat([U[:3], torch.stack(_sym(torch, *U[3:], torch.exp))])
            out.append(U.cpu().numpy())
        return out
    if kind == "gradient":
        ns, ic = _state_of(case, seed)
        S = _Stencils(ns, case["order"])
        U0 = _dev(_registers(ic, "di")).requires_grad_(True)
        Wi, beta = (torch.tensor(v, dtype=torch.float64, device=U0.device, requires_grad=True)
                    for v in (1.0, 0.5))
        M = _Model(S, "di", **dict(GRAD_PHYS, Wi=Wi, beta=beta))
        U, loss = U0.T.contiguous(), 0.0
        for _ in range(case["steps"]):
            U, _e = M.step(U, _dt(case, ns.smax))
            loss = loss + (U[:, 3] + U[:, 5] - 2.0).mean() / case["steps"]
        loss.backward()
        return dict(loss=loss.detach(), U=U0.grad, Wi=Wi.grad.cpu(), beta=beta.grad.cpu())
    if kind == "weights":
        ns, om = _cylinder_of(case, seed)
        S, fields = _Stencils(ns, 8, om), [_field_of(ns, seed)]
    else:
        ns = _lattice(case, seed)
        S = _Stencils(ns, case["order"])
        fields = [_field_of(ns, seed, k) for k in range(case["fields"])]
    F = _dev(np.stack(fields, 1))
    X, Y, L = S.grads(F)
    H = S.filtered(F)
    nf = F.shape[1]
    return dict(grad=[torch.cat([X[:, k], Y[:, k]]) for k in range(nf)],
                lap=[L[:, k].contiguous() for k in range(nf)],
                filt=[H[:, k].contiguous() for k in range(nf)])
