"""Performance cases of the framework: what a program does with it, through
its public entry points, over the sizes it is used at.

A case is one of
  flow   a state uploaded, `steps` time steps run on the device, the state
         downloaded: a run between two outputs or checkpoints
  phase  the same loop driven phase by phase from the host, with the conserved
         integrals after every step (explicitLoop with consCalc): a program
         that couples to the solver, where latency counts
  relax  the phase relaxation alone on states far from equilibrium: a program
         that uses the library for its equilibrium solve
  train  surrogate training on a resident training set
  check  labelling of fresh states and the network's prediction on them

Meshes and network weights are what such a program keeps, so they are built
once per process; the initial states, training sets and sample states come
from the seed.
"""
import functools
import math

import numpy as np
import torch

from fooskagpu_amd import FP64, MIXED, RELAX_COLD, RELAX_MLP, RELAX_PLAIN, GpuSolver, _lib, cases, surrogate
from fooskagpu_amd.mesh import BC_OUTLET, BC_SLIP, BC_WALL, KIND_HEX, Mesh, place_bubbles

PRECISION = {"fp64": FP64, "mixed": MIXED}
RELAX = {"plain": RELAX_PLAIN, "mlp": RELAX_MLP, "cold": RELAX_COLD}
TWO_PI = 2 * math.pi


def listed():
    return [
        # the smallest call: a coupled program on a coarse Sod tube
        dict(name="sod phases 768", kind="phase", flow="sod", nx=8, ny=4, nz=4, precision="fp64", steps=10),
        # the Sod tube of the test matrix as it is run, 100 steps in one call
        dict(name="sod 12288", kind="flow", flow="sod", nx=32, ny=8, nz=8, precision="fp64", steps=100),
        # Taylor-Green vortex on an odd mesh: WALE, viscous terms, heat flux, periodic faces
        dict(name="tgv 23^3", kind="flow", flow="tgv", nx=23, ny=23, nz=23, precision="fp64", steps=40),
        # the 64^3 LES configuration in mixed precision
        dict(name="tgv 64^3 mixed", kind="flow", flow="tgv", nx=64, ny=64, nz=64, precision="mixed", steps=50),
        # bubble collapse, a resolution study's coarse end
        dict(name="bubble 24^3", kind="flow", flow="bubble", nx=24, ny=24, nz=24, precision="fp64", relax="plain",
             steps=20),
        # every element type of a file mesh (tets, pyramids, prisms, hexahedra), viscous
        dict(name="elements 41x17x19", kind="flow", flow="elements", nx=41, ny=17, nz=19, precision="fp64",
             relax="plain", steps=30),
        # shock-bubble on hexahedra, mixed precision, the surrogate pipeline from the cell state
        dict(name="shock hex 72^3 mixed", kind="flow", flow="shock_hex", nx=72, ny=72, nz=72, precision="mixed",
             relax="cold", steps=50),
        # shock-bubble in double precision with the reference's relaxation
        dict(name="shock 56^3", kind="flow", flow="shock", nx=56, ny=56, nz=56, precision="fp64", relax="plain",
             steps=40),
        # the largest: the benchmark's workload (Morton order, WALE, surrogate relaxation), at 3.1M cells
        dict(name="shock 80^3 mixed", kind="flow", flow="shock", nx=80, ny=80, nz=80, precision="mixed", relax="mlp",
             steps=50),
        # equilibrium solve of states far from equilibrium, about a quarter of them chemical
        dict(name="relax 500k", kind="relax", n=500_000, precision="fp64", relax="mlp"),
        # a stretch of surrogate training at the benchmark's batch size
        dict(name="train 8192", kind="train", n=100_000, batch=8192, steps=200),
        # labelling and prediction of fresh states
        dict(name="check 300k", kind="check", n=300_000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["flow"] * 7 + ["phase", "relax", "relax", "train", "check"])
    if kind == "relax":
        return dict(kind="relax", n=_log(rng, 2_000, 1_000_000), precision=rng.choice(["fp64", "mixed"]),
                    relax=rng.choice(["plain", "mlp", "cold"]))
    if kind == "train":
        return dict(kind="train", n=_log(rng, 20_000, 200_000), batch=_log(rng, 100, 16_384), steps=_log(rng, 20, 200))
    if kind == "check":
        return dict(kind="check", n=_log(rng, 1_000, 500_000))
    flow = "sod" if kind == "phase" else rng.choice(["sod", "tgv", "bubble", "elements", "shock_hex", "shock"])
    c = dict(kind=kind, flow=flow)
    if flow == "sod":
        c.update(nx=_log(rng, 6, 64), ny=_log(rng, 3, 12), nz=_log(rng, 3, 12))
    elif flow == "elements":
        c.update(nx=_log(rng, 7, 60), ny=_log(rng, 3, 40), nz=_log(rng, 3, 40))
    else:
        n = _log(rng, 6, 40 if flow == "bubble" else 64)
        c.update(nx=n, ny=n, nz=n if flow == "tgv" else max(5, n - rng.randrange(4)))
    c.update(precision=rng.choice(["fp64", "mixed"]), steps=_log(rng, 5, 20))
    if flow in ("sod", "tgv"):
        c["steps"] *= 1 if kind == "phase" else 3
    else:  # the two-phase scheme loses positivity late in a collapse: short runs
        c["relax"] = rng.choice(["plain", "mlp", "cold"])
    return c


# ---- meshes, constants and initial states ----
BOX = {"sod": ((1.0, 0.25, 0.25), 0.0), "tgv": ((TWO_PI,) * 3, 0.1), "bubble": ((1.0, 1.0, 1.0), 0.1),
       "elements": ((1.0, 0.4, 0.4), 0.1), "shock": ((1.0, 1.0, 1.0), 0.1), "shock_hex": ((1.0, 1.0, 1.0), 0.1)}


@functools.lru_cache(maxsize=32)
def _mesh(flow, nx, ny, nz):
    hi, jitter = BOX[flow]
    lo = (0, 0, 0)
    if flow == "sod":
        return Mesh.box(nx, ny, nz, lo, hi, jitter, 0, bc=(BC_OUTLET, BC_OUTLET) + (BC_SLIP,) * 4)
    if flow == "tgv":
        return Mesh.box(nx, ny, nz, lo, hi, jitter, 1, periodic=(True, True, True), order="morton")
    if flow == "elements":
        return Mesh.mixed_box(nx, ny, nz, lo, hi, jitter, 11,
                              bc=(BC_OUTLET, BC_OUTLET, BC_SLIP, BC_WALL, BC_SLIP, BC_SLIP))
    if flow == "shock_hex":
        return Mesh.box(nx, ny, nz, lo, hi, jitter, 4, bc=(BC_OUTLET,) * 6, order="morton", kinds=KIND_HEX)
    return Mesh.box(nx, ny, nz, lo, hi, jitter, 4, bc=(BC_OUTLET,) * 6, order="rcm" if flow == "bubble" else "morton")


def _params(case):
    flow = case.get("flow")
    if flow == "sod":
        p = dict(cases.BASE, gamma=[1.4, 1.4], cfl=0.3)  # 0.5 amplifies rounding on tetrahedra
    elif flow == "tgv":
        p = dict(cases.BASE, viscFlag=1, turbulence=1, heatFlux=1, dynVisc=[1 / 1600.0] * 2,
                 pRef=1 / (1.4 * 0.1 * 0.1), cfl=0.3)
    else:
        visc = 0 if flow in (None, "bubble") else 1
        p = dict(cases.BASE, model=_lib.MODEL_TWO_PHASE, cfl=0.1, viscFlag=visc, turbulence=visc,
                 **cases.WATER_VAPOUR)
    p["precision"] = PRECISION[case.get("precision", "fp64")]
    p["relaxMode"] = RELAX[case.get("relax", "plain")]
    return p


def _initial(case, p, m, seed):
    """The flow's initial state; strengths, places and sizes vary with the seed."""
    rng = np.random.default_rng(seed)
    flow, am, Tw = case["flow"], p["avfMin"], cases.T_WATER
    if flow == "sod":
        return m.init_sod(1.4, 0.0, rng.uniform(0.45, 0.55), (rng.uniform(0.9, 1.1), 0, 0, 0, rng.uniform(0.9, 1.1)),
                          (0.125, 0, 0, 0, 0.1))
    if flow == "tgv":
        return m.init_tgv(1.4, rng.uniform(0.97, 1.03), 1.0, rng.uniform(0.097, 0.103))
    if flow in ("bubble", "elements"):
        w = BOX[flow][0][1]
        c = (rng.uniform(0.45, 0.55), *(w * rng.uniform(0.45, 0.55, 2)))
        u = (0, 0, 0) if flow == "bubble" else (rng.uniform(2, 4), 0, 0)
        return m.init_regions(p, [dict(kind=0, alphaL=1 - am, p=1e7, T=Tw, u=u),
                                  dict(kind=1, c=c, r=rng.uniform(0.13, 0.16) if flow == "bubble" else 0.15,
                                       alphaL=am, p=2340.0, T=Tw)])
    gL, piL, cvL = p["gamma"][0], p["pInf"][0], p["Cp"][0] / p["gamma"][0]
    p0, p1, rho1 = 1e5, 5e7, 1005.0
    rho0 = (p0 + piL) / (cvL * Tw * (gL - 1))
    u1 = math.sqrt((p1 - p0) * (rho1 - rho0) / (rho0 * rho1))
    regions = [dict(kind=0, alphaL=1 - am, p=p0, T=Tw)]
    for c, r in zip(*place_bubbles(24, (0, 0, 0), (1, 1, 1), 0.03, 0.07, 0.2, int(rng.integers(1, 1 << 30)))):
        regions.append(dict(kind=1, c=tuple(c), r=float(r), alphaL=am, p=2340.0, T=Tw))
    regions.append(dict(kind=2, c=(0.1, 0, 0), alphaL=1 - am, p=p1, T=(p1 + piL) / (cvL * rho1 * (gL - 1)),
                        u=(u1, 0, 0)))
    return m.init_regions(p, regions)


@functools.lru_cache(maxsize=4)
def _cells_for(n):
    """Any mesh of at least n cells: the relaxation is cell by cell."""
    return _mesh("bubble", *[max(2, math.ceil((n / 6) ** (1 / 3)))] * 3)


@functools.lru_cache(maxsize=1)
def _weights():
    """A trained network, as a program loads it: plain NumPy least squares on
    the last layer of a fixed random network, from labels of uniform states."""
    p = _params(dict(kind="relax"))
    with GpuSolver(p) as g:
        x, y = surrogate.finite(*surrogate.Surrogate(g).label(surrogate.uniform_states(20_000, p, seed=1)))
    norm = surrogate.fit_norm(x, y)
    w = surrogate.init_weights(3)
    q = surrogate.unpack(w)
    h = (x - norm[0:3]) / norm[3:6]
    for k in "123":
        h = np.tanh(h @ q["W" + k].T.astype(np.float64) + q["b" + k])
    A = np.concatenate([h, np.ones((len(h), 1))], 1)
    t = (y - norm[6:9]) / norm[9:12]
    sol = np.linalg.solve(A.T @ A + 1e-3 * np.eye(65), A.T @ t)
    w[8576:8768] = sol[:64].T.astype(np.float32).ravel()
    w[8768:] = sol[64].astype(np.float32)
    return w, norm


def _training_set(n, seed):
    """Features and targets over the ranges of the labels; a smooth map with noise."""
    rng = np.random.default_rng(seed)
    x = np.stack([rng.uniform(-3, 7, n), rng.uniform(1.0e6, 2.4e6, n), rng.uniform(0, 1, n)], 1)
    T = 330 + 8 * np.sin(x[:, 0]) + 3e-5 * (x[:, 1] - 1.7e6)
    y = np.stack([T, np.arcsinh(10 ** (0.4 * np.tanh(x[:, 0] / 4) + 0.02 * (T - 280)) / 1e4), x[:, 2] ** 2], 1)
    y += rng.normal(size=y.shape) * [0.5, 0.02, 0.01]
    return x.astype(np.float32), y.astype(np.float32)


def prepare(case, seed):
    p, kind = _params(case), case["kind"]
    st = dict(case=case, kind=kind, params=p)
    if kind in ("flow", "phase"):
        m = _mesh(case["flow"], case["nx"], case["ny"], case["nz"])
        st["U"] = _initial(case, p, m, seed)
        st["solver"] = GpuSolver(p, m, st["U"])
    elif kind == "relax":
        m = _cells_for(case["n"])
        st["U"] = surrogate.uniform_states(m.n_cells, p, seed=seed)
        st["solver"] = GpuSolver(p, m, st["U"])
    else:
        st["solver"] = GpuSolver(p)
    st["net"] = surrogate.Surrogate(st["solver"])
    if kind == "train":
        x, y = _training_set(case["n"], seed)
        st["w"], st["norm"], st["seed"] = surrogate.init_weights(seed), surrogate.fit_norm(x, y), seed
        st["net"].set_data(x, y)
    elif kind == "check":
        st["net"].set_weights(*_weights())
        st["U"] = surrogate.uniform_states(case["n"], p, seed=seed)
    elif case.get("relax") == "mlp":
        st["net"].set_weights(*_weights())
    st["solver"].sync()
    return st


def run(st):
    g, net, case = st["solver"], st["net"], st["case"]
    if st["kind"] == "train":
        net.set_weights(st["w"], st["norm"])
        loss = net.train(case["steps"], batch=case["batch"], lr=2e-3, seed=st["seed"])
        return dict(weights=net.weights()[0], loss=np.array(loss, dtype=np.float32))
    if st["kind"] == "check":
        x, y = net.label(st["U"])
        return dict(x=x, y=y, prediction=net.infer(x))
    g.upload_state(st["U"])
    if st["kind"] == "relax":
        n = g.relaxation(RELAX[case["relax"]])
        return dict(U=g.download_state(), chem=n["n_chem"])
    if st["kind"] == "phase":
        integrals = []
        for s in range(case["steps"]):
            dt = g.explicit_loop_phases(1, s)
            integrals.append(g.cons_calc())
        return dict(U=g.download_state(), integrals=np.array(integrals), dt=dt)
    g.set_clock(0.0, 0.0, 0)
    dt, t = g.run_steps(case["steps"])
    return dict(U=g.download_state(), dt=dt, t=t)


def work(case):
    """Bytes: the host's state in and out, and for each RK stage the state (and
    the stage-0 state of stages 1 and 2) read and written and the mesh's
    connectivity and geometry read once; relaxation reads and writes the
    state once a step."""
    kind = case["kind"]
    if kind == "train":
        return dict(bytes=case["steps"] * (case["batch"] * 32 + 8771 * 24), flops=case["steps"] * case["batch"] * 3 * 17152)
    if kind == "check":
        return dict(bytes=case["n"] * (80 + 24 + 12 + 12), flops=case["n"] * (4000 + 17152))
    if kind == "relax":
        n = 6 * max(2, math.ceil((case["n"] / 6) ** (1 / 3))) ** 3
        return dict(bytes=n * 240, flops=n * 1500)
    hexes, single = case["nx"] * case["ny"] * case["nz"], case["flow"] in ("sod", "tgv")
    cells = hexes * {"shock_hex": 1, "elements": 4}.get(case["flow"], 6)
    faces = cells * {"shock_hex": 3.0, "elements": 2.5}.get(case["flow"], 2.0)
    neq, s = (5 if single else 10), (4 if case["precision"] == "mixed" else 8)
    stage = cells * (8 * neq * (2 + 2 / 3) + 4 * s) + faces * (12 + 7 * s)
    step = 3 * stage + (0 if single else 16 * neq * cells)
    flops = 3 * (faces * (400 if single else 900) + cells * neq * 100)
    return dict(bytes=case["steps"] * step + 16 * neq * cells, flops=case["steps"] * flops)


# ---- the same in 64 bits, in plain torch ----
def exact(case, seed):
    kind, dev = case["kind"], "cuda" if torch.cuda.is_available() else "cpu"
    p = _params(case)
    if kind == "train":
        x, y = _training_set(case["n"], seed)
        norm, w = surrogate.fit_norm(x, y), surrogate.init_weights(seed)
        return dict(weights=_train64(w, norm, x, y, case, seed, dev), loss=None)
    if kind == "check":
        x, y = _label64(p, surrogate.uniform_states(case["n"], p, seed=seed), dev)
        w, norm = _weights()
        return dict(x=x.cpu(), y=None, prediction=_mlp64(w, norm, x).cpu())
    if kind == "relax":
        # the reference solves stop at absolute tolerances, or at their best
        # iterate, where far-off states have no equilibrium: no value in 64
        # bits says what they return
        return None
    m = _mesh(case["flow"], case["nx"], case["ny"], case["nz"])
    if m.n_faces * case["steps"] > 200_000_000:
        return None  # more than about 20 s
    return Flow64(p, m, dev).run(_initial(case, p, m, seed), case["steps"], kind == "phase")


def _batches(n, batch, steps, seed):
    """The sample indices of each step: splitmix64 from the seed, modulo n."""
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + np.arange(1, batch * steps + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    return (z % np.uint64(n)).astype(np.int64).reshape(steps, batch)


def _split64(w, dev):
    return [torch.tensor(np.asarray(v, np.float64), device=dev) for v in surrogate.unpack(w).values()]


def _mlp64(w, norm, x):
    W1, b1, W2, b2, W3, b3, W4, b4 = _split64(w, x.device)
    n = torch.tensor(np.asarray(norm, np.float64), device=x.device)
    h = torch.tanh((x - n[0:3]) / n[3:6] @ W1.T + b1)
    h = torch.tanh(h @ W2.T + b2)
    return (torch.tanh(h @ W3.T + b3) @ W4.T + b4) * n[9:12] + n[6:9]


def _train64(w, norm, x, y, case, seed, dev):
    n = np.asarray(norm, np.float64)
    X = torch.tensor((x - n[0:3]) / n[3:6], device=dev)
    Y = torch.tensor((y - n[6:9]) / n[9:12], device=dev)
    q = _split64(w, dev)
    m, v = [torch.zeros_like(a) for a in q], [torch.zeros_like(a) for a in q]
    for t, idx in enumerate(_batches(len(x), case["batch"], case["steps"], seed), 1):
        i = torch.tensor(idx, device=dev)
        h = [X[i]]
        for k in range(3):
            h.append(torch.tanh(h[-1] @ q[2 * k].T + q[2 * k + 1]))
        d = (h[3] @ q[6].T + q[7] - Y[i]) * (2 / (3 * len(i)))
        grad = [None] * 8
        for k in (3, 2, 1, 0):
            grad[2 * k], grad[2 * k + 1] = d.T @ h[k], d.sum(0)
            if k:
                d = (d @ q[2 * k]) * (1 - h[k] ** 2)
        for j in range(8):
            m[j] = 0.9 * m[j] + 0.1 * grad[j]
            v[j] = 0.999 * v[j] + 0.001 * grad[j] ** 2
            q[j] = q[j] - 2e-3 * (m[j] / (1 - 0.9 ** t)) / (torch.sqrt(v[j] / (1 - 0.999 ** t)) + 1e-8)
    return torch.cat([a.reshape(-1) for a in q]).cpu()


def _label64(p, U, dev):
    U = torch.tensor(U, device=dev)
    rho = U[:, 1] + U[:, 2]
    ke = 0.5 * (U[:, 3:6] ** 2).sum(1) / rho
    return torch.stack([torch.log(rho), (U[:, 8] - ke) / rho, U[:, 1] / rho], 1), None


class Flow64:
    """The explicit step on faces: Green-Gauss gradients, limiter, MUSCL, HLLC,
    viscous and WALE terms, SSP-RK3, phase equilibrium."""

    def __init__(self, p, m, dev):
        t = lambda a: torch.tensor(a, device=dev)  # noqa: E731
        self.p, self.two = p, p["model"] == _lib.MODEL_TWO_PHASE
        self.iu = 3 if self.two else 1
        self.o, nb = t(m.fc2el[:, 0].astype(np.int64)), t(m.fc2el[:, 1].astype(np.int64))
        self.inner = nb >= 0
        self.nb = torch.where(self.inner, nb, self.o)
        self.w = self.inner.double()[:, None]  # 1 on interior faces
        self.bc, self.n, self.A, self.V = t(m.bc)[:, None], t(m.n), t(m.area)[:, None], t(m.volume)[:, None]
        xc, xf = t(m.cell_center), t(m.fc_center)
        self.ro, self.rn = xf - xc[self.o], xf - t(m.shift) - xc[self.nb]
        self.Ls = 0.325 * ((self.V[self.o] + self.V[self.nb]) / 2) ** (1 / 3)

    def eos(self, k):
        p = self.p
        g, pi, cv = p["gamma"][k], p["pInf"][k], p["Cp"][k] / p["gamma"][k]
        return g, pi, cv, (p["eta"][k] if self.two else 0.0)

    def press(self, k, rho, e):
        g, pi, _, eta = self.eos(k)
        return (g - 1) * rho * (e - eta) - g * pi

    def energy(self, k, pr, rho):
        g, pi, _, eta = self.eos(k)
        return (pr + g * pi) / (rho * (g - 1)) + eta

    def c2(self, k, rho, pr):
        g, pi, _, _ = self.eos(k)
        return g * (pr + pi) / rho

    def prims(self, U):
        if not self.two:
            u = U[:, 1:4] / U[:, :1]
            return torch.cat([U[:, :1], u, self.press(0, U[:, :1], U[:, 4:] / U[:, :1] - 0.5 * (u * u).sum(1, True))], 1)
        am = self.p["avfMin"] / 100
        a = U[:, :1].clamp(am, 1 - am)
        rl, rg = U[:, 1:2] / a, U[:, 2:3] / (1 - a)
        rm = U[:, 1:2] + U[:, 2:3]
        return torch.cat([a, rl, rg, U[:, 3:6] / rm, self.press(0, rl, U[:, 6:7] / U[:, 1:2]),
                          self.press(1, rg, U[:, 7:8] / U[:, 2:3]), U[:, 9:], rm], 1)

    def ghost(self, W):
        u = W[:, self.iu:self.iu + 3]
        slip = u - 2 * (u * self.n).sum(1, True) * self.n
        u = torch.where((self.bc == 1) | (self.bc == 4), slip, torch.where(self.bc == 5, -u, u))
        return torch.cat([W[:, :self.iu], u, W[:, self.iu + 3:]], 1)

    def gather(self, to_owner, to_neighbour):
        out = torch.zeros(len(self.V), to_owner.shape[1], dtype=torch.float64, device=to_owner.device)
        return out.index_add_(0, self.o, to_owner).index_add_(0, self.nb, to_neighbour * self.w)

    def extreme(self, how, to_owner, to_neighbour):
        out = torch.full((len(self.V), to_owner.shape[1]), -math.inf if how == "amax" else math.inf,
                         dtype=torch.float64, device=to_owner.device)
        e = lambda i, v: i[:, None].expand_as(v)  # noqa: E731
        out.scatter_reduce_(0, e(self.o, to_owner), to_owner, how)
        v = to_neighbour[self.inner]
        return out.scatter_reduce_(0, e(self.nb[self.inner], v), v, how)

    def faces(self, W):
        """Reconstructed states of both sides, velocity (and temperature) gradients."""
        L, R = W[self.o], torch.where(self.inner[:, None], W[self.nb], self.ghost(W[self.o]))
        f = (L + R) / 2 * self.A
        g = [self.gather(f * self.n[:, d:d + 1], -f * self.n[:, d:d + 1]) / self.V for d in range(3)]
        mx, mn = self.extreme("amax", R, L), self.extreme("amin", R, L)

        def side(i, r):
            ext = r[:, :1] * g[0][i] + r[:, 1:2] * g[1][i] + r[:, 2:] * g[2][i]
            d = torch.where(ext > 0, mx[i] - W[i], mn[i] - W[i])
            return ext, torch.where(ext == 0, torch.ones_like(ext), d / (2 * ext)).clamp(0, 1)

        eo, po = side(self.o, self.ro)
        en, pn = side(self.nb, self.rn)
        th = self.extreme("amin", po, pn)
        L = W[self.o] + th[self.o] * eo
        R = torch.where(self.inner[:, None], W[self.nb] + th[self.nb] * en, self.ghost(L))
        iu = self.iu
        G = torch.stack([x[:, iu:iu + 3] for x in g], 2)
        GT = None
        if not self.two:
            _, pi, cv, _ = self.eos(0)
            R0 = cv * (self.p["gamma"][0] - 1)
            GT = torch.stack([(x[:, 4] - (W[:, 4] + pi) / W[:, 0] * x[:, 0]) / (W[:, 0] * R0) for x in g], 1)
        return L, R, G, GT

    def mix(self, s):
        """Mixture density and pressure of face states."""
        if not self.two:
            return s[:, :1], s[:, 4:5]
        a = s[:, :1]
        return a * s[:, 1:2] + (1 - a) * s[:, 2:3], a * s[:, 6:7] + (1 - a) * s[:, 7:8]

    def sound(self, s, wood):
        if not self.two:
            return torch.sqrt(self.c2(0, s[:, :1], s[:, 4:5]))
        a, rl, rg = s[:, :1], s[:, 1:2], s[:, 2:3]
        rm = a * rl + (1 - a) * rg
        cl, cg = self.c2(0, rl, s[:, 6:7]), self.c2(1, rg, s[:, 7:8])
        return torch.where(wood, 1 / torch.sqrt(rm * (a / (rl * cl) + (1 - a) / (rg * cg))),
                           torch.sqrt((a * rl * cl + (1 - a) * rg * cg) / rm))

    def wood(self, y):
        return (y > self.p["chemLimit"]) & (self.p["woodsFlag"] == 1)

    def residual(self, U):
        W, n, iu = self.prims(U), self.n, self.iu
        L, R, G, GT = self.faces(W)
        dot = lambda s: (s[:, iu:iu + 3] * n).sum(1, True)  # noqa: E731
        uL, uR = dot(L), dot(R)
        y = (L[:, 8:9] + R[:, 8:9]) / 2 if self.two else L[:, :1]
        cL, cR = self.sound(L, self.wood(y)), self.sound(R, self.wood(y))
        S0, S2 = torch.minimum(uL - cL, uR - cR), torch.maximum(uL + cL, uR + cR)
        (rL, pL), (rR, pR) = self.mix(L), self.mix(R)
        S1 = (pR - pL + rL * uL * (S0 - uL) - rR * uR * (S2 - uR)) / (rL * (S0 - uL) - rR * (S2 - uR))
        S1 = torch.where(self.bc == 5, torch.zeros_like(S1), S1)
        left, star = S1 >= 0, (S0 < 0) & (S2 >= 0)
        s, un, SK = torch.where(left, L, R), torch.where(left, uL, uR), torch.where(left, S0, S2)
        rho, pr = self.mix(s)
        u = s[:, iu:iu + 3]
        ke = 0.5 * (u * u).sum(1, True)
        us = torch.where(star, u + (S1 - un) * n, u)  # velocity of the star region
        k = (SK - un) / (SK - S1)
        H = lambda v: torch.where(star, SK * v, torch.zeros_like(v))  # noqa: E731
        if not self.two:
            E = rho * (self.energy(0, pr, rho) + ke)
            Es = k * (E + rho * (S1 - un) * (S1 + pr / (rho * (SK - un))))
            f = torch.cat([rho * un + H(rho * k - rho), rho * un * u + pr * n + H(rho * k * us - rho * u),
                           (E + pr) * un + H(Es - E)], 1)
            to_o, to_n = -f * self.A, f * self.A
        else:
            a, rl, rg = s[:, :1], s[:, 1:2], s[:, 2:3]
            el, eg = self.energy(0, s[:, 6:7], rl), self.energy(1, s[:, 7:8], rg)
            E = a * rl * el + (1 - a) * rg * eg + rho * ke
            gl, pil, _, _ = self.eos(0)
            gg, pig, _, _ = self.eos(1)
            ps = lambda g, pi, q, r: (q + pi) * ((g - 1) - (g + 1) * k) / ((g - 1) * k - (g + 1)) - pi  # noqa: E731
            al = a * torch.where(star, rl * k * self.energy(0, ps(gl, pil, s[:, 6:7], rl), rl * k), rl * el)
            ag = (1 - a) * torch.where(star, rg * k * self.energy(1, ps(gg, pig, s[:, 7:8], rg), rg * k), rg * eg)
            V8 = k * (E + (S1 - un) * (S1 + pr / (rho * (SK - un))))
            usn = (us * n).sum(1, True)
            fl = [usn * a, un * a * rl + H(a * rl * (k - 1)), un * (1 - a) * rg + H((1 - a) * rg * (k - 1)),
                  rho * un * u + H(rho * k * us - rho * u), usn * al, usn * ag,
                  un * (E + pr) + H(V8 - E), un * s[:, 8:9] + H(s[:, 8:9] * (k - 1))]

            def side(i):
                ac, pl, pg = W[i, :1], W[i, 6:7], W[i, 7:8]
                return torch.cat([fl[0] - ac * usn, fl[1], fl[2], fl[3] + (pr - (ac * pl + (1 - ac) * pg)) * n,
                                  fl[4] + ac * pl * usn, fl[5] + (1 - ac) * pg * usn, fl[6], fl[7]], 1) * self.A

            to_o, to_n = -side(self.o), side(self.nb)
        if self.p["viscFlag"]:
            v = self.viscous(W, L, R, G, GT)
            to_o, to_n = to_o + v, to_n - v
        yl, yr = (L[:, 8:9], R[:, 8:9]) if self.two else (y, y)
        sig = uL.abs() + self.sound(L, self.wood(yl))
        sig = torch.maximum(sig, (uR.abs() + self.sound(R, self.wood(yr))) * self.w)
        return self.gather(to_o, to_n), self.extreme("amax", sig, sig)

    def viscous(self, W, L, R, G, GT):
        """Owner-side viscous contribution n.tau A of each equation."""
        gm = (G[self.o] + G[self.nb]) / 2
        eye = torch.eye(3, dtype=torch.float64, device=gm.device)
        tr = torch.diagonal(gm, dim1=1, dim2=2).sum(1)[:, None, None]
        st = gm + gm.transpose(1, 2) - 2 / 3 * tr * eye
        mu = self.p["dynVisc"]
        R1 = torch.where(self.inner[:, None], R, self.ghost(W[self.o]))
        rhof = (self.mix(L)[0] + self.mix(R1)[0]) / 2
        nu = torch.zeros_like(rhof)
        if self.p["turbulence"]:
            sq = gm @ gm
            sd = (sq + sq.transpose(1, 2)) / 2 - torch.diagonal(sq, dim1=1, dim2=2).sum(1)[:, None, None] / 3 * eye
            a = (sd * sd).sum((1, 2))[:, None]
            b = (((gm + gm.transpose(1, 2)) / 2) ** 2).sum((1, 2))[:, None]
            den = a ** 1.25 + b ** 2.5 + 1e-12
            nu = torch.where(den < 1e-10, torch.zeros_like(a), self.Ls ** 2 * a ** 1.5 / den)
        if self.two:
            af = (L[:, :1] + R1[:, :1]) / 2
            mu = af * mu[0] + (1 - af) * mu[1] + rhof * nu
        else:
            mu = mu[0] + rhof * nu
        fm = mu * (st * self.n[:, None, :]).sum(2)
        uf = (L[:, self.iu:self.iu + 3] + R1[:, self.iu:self.iu + 3]) / 2
        fe = mu * ((st * uf[:, None, :]).sum(2) * self.n).sum(1, True)
        out = torch.zeros_like(L)
        out[:, self.iu:self.iu + 3] = fm * self.A
        if self.two:
            out[:, 8:9] = fe * self.A
        else:
            gt = (GT[self.o] + GT[self.nb]) / 2
            out[:, 4:5] = (fe + self.p["Cp"][0] * mu / self.p["Pr"][0] * (gt * self.n).sum(1, True)) * self.A
        return out

    def relax(self, U):
        """Pressure and temperature equilibrium of every cell: with the mass and
        energy balances a quadratic in p.  Cells with superheated liquid also
        reach equal Gibbs energies."""
        p = self.p
        (gl, pl, cl, el), (gg, pg, cg, eg) = self.eos(0), self.eos(1)
        al, ag = U[:, 1], U[:, 2]
        E = U[:, 8] - 0.5 * (U[:, 3:6] ** 2).sum(1) / (al + ag)
        W = self.prims(U)
        TL = (W[:, 6] + pl) / (cl * (gl - 1) * W[:, 1])
        chem = (W[:, 0] > p["chemLimit"]) & (self.saturation(W[:, 6], TL) > 0)
        A, B, E1 = (al * cl * (gl - 1), ag * cg * (gg - 1)), (al * cl, ag * cg), E - al * el - ag * eg
        q2 = B[0] + B[1]
        q1 = B[0] * (gl * pl + pg) + B[1] * (gg * pg + pl) - E1 * (A[0] + A[1])
        q0 = B[0] * gl * pl * pg + B[1] * gg * pg * pl - E1 * (A[0] * pg + A[1] * pl)
        root = torch.sqrt((q1 * q1 - 4 * q2 * q0).clamp(min=0))
        pr = torch.where(q1 < 0, (root - q1) / (2 * q2), -2 * q0 / (q1 + root))
        T = 1 / (A[0] / (pr + pl) + A[1] / (pr + pg))
        if bool(chem.any()):
            i = chem.nonzero()[:, 0]
            pc, Tc = self.gibbs(al[i] + ag[i], E[i], TL[i], W[i, 6].clamp(min=1e3))
            rl, rg = (pc + pl) / (cl * (gl - 1) * Tc), (pc + pg) / (cg * (gg - 1) * Tc)
            a = (al[i] + ag[i] - rg) / (rl - rg)
            ok = (a > 0) & (a < 1) & torch.isfinite(a)
            i, pr[i[ok]], T[i[ok]] = i[ok], pc[ok], Tc[ok]
            al, ag = al.clone(), ag.clone()
            al[i], ag[i] = (a * rl)[ok], ((1 - a) * rg)[ok]
            U = U.clone()
            U[:, 1], U[:, 2] = al, ag
            U[i, 9] = ag[i]
        e = [cv * T * (pr + g * pi) / (pr + pi) + eta for g, pi, cv, eta in (self.eos(0), self.eos(1))]
        am = p["avfMin"] / 100
        a = (al * cl * (gl - 1) * T / (pr + pl)).clamp(am, 1 - am)
        return torch.cat([a[:, None], U[:, 1:6], (al * e[0])[:, None], (ag * e[1])[:, None], U[:, 8:]], 1)

    def saturation(self, pr, T):
        """Positive where the liquid is superheated: the Gibbs difference over T."""
        p = self.p
        d = p["Cp"][1] - self.eos(1)[2]
        cp, et = p["Cp"], p["satConst"][0] * torch.log10(pr) + p["satConst"][1]
        return (cp[0] - cp[1] + et + (p["eta"][0] - p["eta"][1]) / T + (cp[1] - cp[0]) * torch.log10(T)
                + (cp[0] - self.eos(0)[2]) * torch.log10(pr + p["pInf"][0])) / d - torch.log10(pr)

    def gibbs(self, rho, E, T, pr):
        """(p, T) of the two-phase equilibrium at (rho, rho e): Newton with
        differenced Jacobian in (ln p, T), steps limited."""
        def res(lp, T):
            q = torch.exp(lp)
            r, en, gi = [], [], []
            for k in (0, 1):
                g, pi, cv, eta = self.eos(k)
                r.append((q + pi) / (cv * (g - 1) * T))
                en.append((q + g * pi) / (g - 1) + eta * r[k])
                et = 0.0 if k == 0 else self.p["satConst"][0] * torch.log10(q) + self.p["satConst"][1]
                gi.append(g * cv * T + eta - T * (cv * (g * torch.log10(T) - (g - 1) * torch.log10(q + pi)) + et))
            a = (rho - r[1]) / (r[0] - r[1])
            return (en[1] + a * (en[0] - en[1]) - E) / 1e6, (gi[0] - gi[1]) / 1e4
        lp = torch.log(pr)
        for _ in range(60):
            f, g = res(lp, T)
            (fp, gp), (fq, gq) = res(lp + 1e-6, T), res(lp - 1e-6, T)
            (ft, gt), (fs, gs) = res(lp, T + 1e-4), res(lp, T - 1e-4)
            a, b, c, d = (fp - fq) / 2e-6, (ft - fs) / 2e-4, (gp - gq) / 2e-6, (gt - gs) / 2e-4
            det = a * d - b * c
            dl, dT = (d * f - b * g) / det, (a * g - c * f) / det
            lim = torch.maximum(dl.abs(), dT.abs() / (0.2 * T)).clamp(min=1)
            lp, T = lp - dl / lim, T - dT / lim
        return torch.exp(lp), T

    def run(self, U, steps, phases):
        U = torch.tensor(U, device=self.V.device)
        p, t, integrals = self.p, 0.0, []
        for _ in range(steps):
            U0 = U
            for irk, (a, b) in enumerate(((0.0, 1.0), (0.75, 0.25), (1 / 3, 2 / 3))):
                rhs, sig = self.residual(U)
                if irk == 0:
                    dt = min(p["cfl"] * float((self.V ** 0.3333 / sig).min()), p["maxDt"])
                U = a * U0 + b * (U + dt * rhs / self.V)
            t += dt
            if self.two:
                U = self.relax(U)
            if phases:
                q = torch.cat([1 - U[:, :1], U[:, 1:]], 1) if self.two else U
                integrals.append((q * self.V).sum(0).cpu())
        if phases:
            return dict(U=U.cpu(), integrals=torch.stack(integrals), dt=dt)
        return dict(U=U.cpu(), dt=dt, t=t)
