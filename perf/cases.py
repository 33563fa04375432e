"""Performance cases of the heat path: the work that programs on this library
have it do, through its public entry points, over the range of sizes that the
workloads, inputs and tests of this repository use.

Kinds of cases:

``vmult``     one operator application (ThermalOperatorDevice.vmult)
``steps``     explicit time steps of one operator (ThermalPhysicsDevice.evolve)
``ensemble``  explicit time steps of an ensemble (EnsembleDevice.evolve)
``gradient``  misfit and gradient of one operator (adjoint_gradient)
``gradients`` the same for every member (ensemble_adjoint_gradient)
``analysis``  one EnKF analysis (DataAssimilator.update_ensemble)

Materials: ``solid`` is one solid state with polynomial properties and no
boundary term (workloads.plain_small); ``slp`` is solid/liquid/powder with
tabulated properties, latent heat and a convective and radiative top
(workloads.plain_large); ``deposit`` is the same material under an electron
beam with the lowest tenth of the cell layers active
(workloads.deposition_workload). Temperatures are a melt pool under the beam
over a gently varying plate, as a scan leaves them. Stepping cases start each
pass from the same temperatures, as a calibration does.

``exact`` restates the weak form, the phase model, the heat sources, the time
steppers, the adjoint (by torch's autograd) and the Kalman update in float64
torch, cell by cell, with none of the library's code.
"""
import math

import numpy as np
import torch

from adamantine_amd import workloads
from adamantine_amd.adjoint import adjoint_gradient, ensemble_adjoint_gradient
from adamantine_amd.ensemble import DataAssimilator, EnsembleDevice, Member
from adamantine_amd.problem import (FORWARD_EULER, RK_FOURTH_ORDER,
                                    RK_THIRD_ORDER, SOURCE_GOLDAK)
from adamantine_amd.thermal import ThermalOperatorDevice, ThermalPhysicsDevice

METHODS = {"fe": FORWARD_EULER, "rk3": RK_THIRD_ORDER, "rk4": RK_FOURTH_ORDER}
STAGES = {"fe": 1, "rk3": 3, "rk4": 4}
STEFAN_BOLTZMANN = 5.670374419e-8


def _case(name, kind, material, degree, cells, **more):
    c = {"name": name, "kind": kind, "material": material, "degree": degree,
         "nx": cells[0], "ny": cells[1], "nz": cells[2]}
    c.update(more)
    return c


def listed():
    return [
        # the smallest calls: steps of the 5,049-node box on which a user
        # tries an input out
        _case("steps_q1_small", "steps", "solid", 1, (32, 16, 8),
              method="fe", n_steps=10, dt=1e-6),
        # the headline operator and its time step, 2.15 million nodes
        _case("vmult_q2_large", "vmult", "slp", 2, (128, 64, 32)),
        _case("steps_q2_large", "steps", "slp", 2, (128, 64, 32),
              method="rk4", n_steps=2, dt=5e-7),
        # one simulation of ordinary size: the member of an ensemble run on
        # its own, with its top cell layers still inactive
        _case("steps_q2_member", "steps", "slp", 2, (64, 32, 16),
              active=12, method="rk4", n_steps=5, dt=5e-7),
        # degree 3, which most of the input files ask for, at a ragged size
        _case("steps_q3", "steps", "slp", 3, (50, 25, 17),
              method="rk4", n_steps=1, dt=2e-7),
        # the right-hand side of a user's own integrator on linear elements,
        # with every feature of the material, at a ragged size
        _case("vmult_q1_ragged", "vmult", "slp", 1, (101, 67, 33)),
        # a filter's forecast: every member of the ensemble one step on
        _case("ensemble_q2", "ensemble", "slp", 2, (64, 32, 16),
              members=64, method="rk4", n_steps=1, dt=5e-7),
        # a deposition ensemble early in its build
        _case("ensemble_deposit", "ensemble", "deposit", 2, (96, 96, 40),
              members=8, method="fe", n_steps=10, dt=2e-7),
        # one gradient of a calibration
        _case("gradient_q2", "gradient", "slp", 2, (64, 32, 16), active=12,
              method="rk4", n_steps=20, dt=5e-7, every=10, n_obs=200),
        # every member's gradient of a calibration ensemble
        _case("gradients_q2", "gradients", "slp", 2, (48, 24, 16),
              members=8, method="fe", n_steps=20, dt=5e-7, every=10,
              n_obs=200),
        # a filter's analysis: every observation acts on every node
        _case("analysis_global", "analysis", "slp", 2, (64, 32, 16),
              members=64, n_obs=500, localization="none", cutoff=1e3),
        # the same with localised covariances, as the input files ask for
        _case("analysis_local", "analysis", "slp", 2, (64, 32, 16),
              members=32, n_obs=200, localization="gaspari_cohn",
              cutoff=1e-3),
    ]


def draw(rng):
    def log_int(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(
            math.log(lo - 0.499), math.log(hi + 0.499)))))))

    def box(scale_x, scale_y, scale_z):
        f = rng.uniform(0.0, 1.0)  # the box's size, one factor for the axes
        def axis(lo, hi):
            n = lo * (hi / lo) ** min(1.0, max(0.0, f + rng.uniform(-0.1, 0.1)))
            return max(lo, min(hi, int(round(n))))
        return axis(*scale_x), axis(*scale_y), axis(*scale_z)

    kind = rng.choice(["vmult", "vmult", "steps", "steps", "steps",
                       "ensemble", "ensemble", "gradient", "gradients",
                       "analysis"])
    if kind in ("vmult", "steps"):
        degree = rng.choice([1, 2, 2, 3])
        top = {1: (128, 64, 32), 2: (128, 64, 32), 3: (64, 32, 20)}[degree]
        material = rng.choice(["solid", "slp", "slp"]) if degree < 3 else "slp"
        cells = box((24, top[0]), (12, top[1]), (8, top[2]))
        more = {}
        if material == "slp" and rng.random() < 0.5:
            more["active"] = rng.randint(max(5, cells[2] // 2), cells[2])
        if kind == "steps":
            more.update(method=rng.choice(["fe", "rk3", "rk4"]),
                        n_steps=rng.randint(1, 4), dt=2e-7)
            if degree > 2:
                more["n_steps"] = rng.randint(1, 2)
            elif cells[0] * cells[1] * cells[2] > 130000:
                more["n_steps"] = rng.randint(1, 2)
        return _case("", kind, material, degree, cells, **more)
    if kind == "ensemble":
        if rng.random() < 0.4:
            nz = 10 * rng.randint(1, 4)
            cells = (rng.randint(32, 96), rng.randint(32, 96), nz)
            return _case("", kind, "deposit", 2, cells,
                         members=rng.randint(2, 8), method="fe",
                         n_steps=rng.randint(2, 10), dt=2e-7)
        cells = box((16, 64), (8, 32), (8, 16))
        return _case("", kind, "slp", rng.choice([1, 2, 2, 2]), cells,
                     members=log_int(2, 64),
                     method=rng.choice(["fe", "rk4", "rk4"]), n_steps=1,
                     dt=5e-7)
    if kind == "gradient":
        cells = box((16, 64), (8, 32), (8, 16))
        steps = rng.randint(4, 20)
        return _case("", kind, "slp", rng.choice([1, 2, 2]), cells,
                     active=rng.randint(max(5, cells[2] // 2), cells[2]),
                     method=rng.choice(["fe", "rk3", "rk4"]), n_steps=steps,
                     dt=5e-7, every=rng.randint(2, steps),
                     n_obs=log_int(20, 300))
    if kind == "gradients":
        cells = box((16, 48), (8, 24), (8, 16))
        steps = rng.randint(4, 20)
        return _case("", kind, "slp", 2, cells, members=rng.randint(2, 8),
                     method="fe", n_steps=steps, dt=5e-7,
                     every=rng.randint(2, steps), n_obs=log_int(20, 300))
    cells = box((16, 64), (8, 32), (8, 16))
    fn = rng.choice(["none", "gaspari_cohn", "step_function"])
    members = log_int(3, 64)
    most = max(20, min(200, 200 * 32 // members))
    return _case("", kind, "slp", rng.choice([1, 2, 2]), cells,
                 members=members, n_obs=log_int(20, most), localization=fn,
                 cutoff=rng.uniform(0.5e-3, 2e-3))


# ---------------------------------------------------------------------------
# what a program has before the call
# ---------------------------------------------------------------------------

def _cells(c):
    return (c["nx"], c["ny"], c["nz"])


def _problem(c):
    """The problem, and the members for the ensemble kinds (else None)."""
    members = None
    if c["material"] == "solid":
        p = workloads.plain_small(n_cells=_cells(c))
    elif c["material"] == "deposit":
        w = workloads.deposition_workload(n_members=c["members"],
                                          n_cells=_cells(c))
        p, members = w.base, w.members
    elif "members" in c:
        p, members = workloads.ensemble_workload(n_members=c["members"],
                                                 n_cells=_cells(c))
    else:
        p = workloads.plain_large(n_cells=_cells(c))
        if c.get("active", c["nz"]) < c["nz"]:
            top = c["active"] * p.extent[2] / c["nz"]
            p.beams[0].segments = workloads.serpentine(z=top)
            p.set_material_height(top)
            p.set_powder_layer(top, 4 * p.extent[2] / c["nz"])
    p.fe_degree = c["degree"]
    p.method = METHODS[c.get("method", "rk4")]
    return p, members


def _start_time(p, rng):
    """A moment of the beam's first track."""
    segs = p.beams[0].segments
    on = next(k for k, s in enumerate(segs) if s[1] > 0.0)
    t0 = segs[on - 1][0]
    return t0 + rng.uniform(0.2, 0.6) * (segs[on][0] - t0)


def _axes(p):
    """The node coordinates along each axis."""
    xs = _lobatto(p.fe_degree)[0]
    out = []
    for a in range(3):
        h = p.extent[a] / p.n_cells[a]
        x = [(k + v) * h for k in range(p.n_cells[a]) for v in xs[:-1]]
        out.append(torch.tensor(x + [p.extent[a]], dtype=torch.float64,
                                device="cuda"))
    return out


def _field(p, t, rng, n=1):
    """[n, nodes] temperatures: a plate around 350 K with a melt pool under
    the beam."""
    x, y, z = _axes(p)
    cx, cy, cz = _beam_at(p, t)[0]
    L = p.extent
    out = torch.empty((n, p.n_dofs), dtype=torch.float64, device="cuda")
    for j in range(n):
        peak, amb = rng.uniform(1900.0, 2800.0), rng.uniform(320.0, 380.0)
        sx, sy = rng.uniform(110e-6, 190e-6), rng.uniform(90e-6, 150e-6)
        sz, ph = rng.uniform(60e-6, 100e-6), rng.uniform(0.0, 6.0)
        ex = torch.exp(-(x - cx) ** 2 / (2 * sx * sx))
        ey = torch.exp(-(y - cy) ** 2 / (2 * sy * sy))
        ez = torch.exp(-(z - cz) ** 2 / (2 * sz * sz))
        f = (peak - amb) * ez[:, None, None] * ey[None, :, None] * ex
        f += amb + 12.0 * torch.sin(3.0 * x / L[0] + ph)
        f += 9.0 * torch.cos(4.0 * y / L[1] + ph)[None, :, None]
        f += 7.0 * torch.sin(5.0 * z / L[2] - ph)[:, None, None]
        out[j] = f.reshape(-1)
    return out


def _top_nodes(p, active_layers, count, rng):
    """Distinct nodes of the scanned surface around the tracks."""
    nn = p.n_nodes
    iz = p.fe_degree * active_layers
    ix = np.arange(int(0.1 * nn[0]), int(0.9 * nn[0]))
    iy = np.arange(int(0.35 * nn[1]), max(int(0.65 * nn[1]),
                                          int(0.35 * nn[1]) + 3))
    pick = rng.permutation(ix.size * iy.size)[:count]
    return np.sort(ix[pick % ix.size] +
                   nn[0] * (iy[pick // ix.size] + nn[1] * iz)).astype(np.int64)


def _inputs(c, seed):
    """The seed's inputs, as prepare and exact both use them."""
    rng = np.random.RandomState(seed % (2 ** 31))
    p, members = _problem(c)
    t = _start_time(p, rng)
    s = {"problem": p, "members": members, "t": t}
    if c["kind"] == "analysis":
        N = len(members)
        mean = _field(p, t, rng)[0]
        x, y, z = _axes(p)
        X = torch.empty((N, p.n_dofs), dtype=torch.float64, device="cuda")
        for j in range(N):
            a, b, d = rng.uniform(0.0, 6.0, 3)
            k = rng.uniform(2.0, 12.0, 3)
            w = torch.sin(k[0] * x / p.extent[0] + a)
            w = torch.cos(k[1] * y / p.extent[1] + b)[:, None] * w
            w = torch.sin(k[2] * z / p.extent[2] + d)[:, None, None] * w
            X[j] = mean + rng.normal(0.0, 15.0) + 20.0 * w.reshape(-1)
        obs = _top_nodes(p, (3 * c["nz"]) // 4, c["n_obs"], rng)
        m = obs.size
        at = torch.tensor(obs, device="cuda")
        s.update(X=X, obs=obs,
                 y=mean[at].cpu().numpy() + rng.normal(0.0, 2.0, m),
                 R=4.0 * np.eye(m), noise=rng.normal(0.0, 2.0, (N, m)),
                 params=np.ascontiguousarray(rng.normal(
                     [0.3, 1.0], [0.05, 0.1], (N, 2))))
        return s
    s["T"] = _field(p, t, rng, len(members) if members else 1)
    if c["kind"] in ("gradient", "gradients"):
        layers = c.get("active", (3 * c["nz"]) // 4)
        obs = _top_nodes(p, layers, c["n_obs"], rng)
        at = torch.tensor(obs, device="cuda")
        val = s["T"][:, at].cpu().numpy()
        s.update(obs=obs, y=val + rng.normal(0.0, 20.0, val.shape))
    return s


def _node_points(p, nodes):
    x = [a.cpu().numpy() for a in _axes(p)]
    nn = p.n_nodes
    return np.stack([x[0][nodes % nn[0]], x[1][(nodes // nn[0]) % nn[1]],
                     x[2][nodes // (nn[0] * nn[1])]], axis=1)


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    p, kind = s["problem"], case["kind"]
    if kind == "vmult":
        s["op"] = ThermalOperatorDevice(p)
        s["op"].set_time(s["t"])
        s["T"] = s["T"][0]
        s["dst"] = s["op"].initialize_dof_vector()
    elif kind in ("steps", "gradient"):
        s["ph"] = ThermalPhysicsDevice(p)
        s["ph"].setup()
        s["T"] = s["T"][0]
    else:
        s["ens"] = EnsembleDevice(p, s["members"])
        s["ens"].compute_inverse_mass_matrix()
    if kind in ("steps", "ensemble"):
        s["sol"] = torch.empty_like(s["T"])
    if kind == "analysis":
        s["da"] = DataAssimilator(case["localization"], case["cutoff"])
        s["da"].update_dof_mapping(s["ens"], _node_points(p, s["obs"]))
        s["sol"] = torch.empty_like(s["X"])
    return s


def run(state):
    c, kind = state["case"], state["case"]["kind"]
    if kind == "vmult":
        state["op"].vmult(state["dst"], state["T"])
        return state["dst"]
    if kind == "steps":
        state["sol"].copy_(state["T"])
        state["ph"].evolve(state["t"], c["dt"], c["n_steps"], state["sol"])
        return state["sol"]
    if kind == "ensemble":
        state["sol"].copy_(state["T"])
        state["ens"].evolve(state["t"], c["dt"], c["n_steps"], state["sol"])
        return state["sol"]
    if kind == "gradient":
        r = adjoint_gradient(state["ph"], state["t"], c["dt"], c["n_steps"],
                             state["T"], state["obs"], state["y"][0],
                             checkpoint_every=c["every"])
        return {"J": r.J, "grad": r.grad, "T_final": r.T_final,
                "lambda0": r.lambda0}
    if kind == "gradients":
        r = ensemble_adjoint_gradient(
            state["ens"], state["t"], c["dt"], c["n_steps"], state["T"],
            state["obs"], state["y"], checkpoint_every=c["every"])
        return {"J": r.J, "grad": r.grad, "T_final": r.T_final,
                "lambda0": r.lambda0}
    state["sol"].copy_(state["X"])
    params = state["params"].copy()
    state["da"].update_ensemble(state["ens"], state["sol"], state["y"],
                                state["R"], params=params,
                                noise=state["noise"])
    return {"X": state["sol"], "params": params}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _layers(c):
    """Active cell layers, summed over the members."""
    if c["material"] == "deposit":
        return c["members"] * (c["nz"] // 10)
    if "members" in c:
        base = (3 * c["nz"]) // 4
        return sum(min(base + j % 5, c["nz"]) for j in range(c["members"]))
    return c.get("active", c["nz"])


def work(case):
    N = case["degree"] + 1
    nodes = 1
    for n in _cells(case):
        nodes *= case["degree"] * n + 1
    members = case.get("members", 1)
    cells = case["nx"] * case["ny"] * _layers(case)
    kind = case["kind"]
    if kind == "analysis":
        # read and written once; per node the member mean and anomalies, and
        # with m observations 2 m N to form the covariances and 2 m N to
        # apply them (localised), or an N x N transform
        m = case["n_obs"]
        per = 4 * m * members if case["localization"] != "none" else \
            2 * members * members
        return {"bytes": 16.0 * nodes * members + 8.0 * m * (members + m),
                "flops": float(nodes) * per}
    # nodes that an active cell holds, at most
    layers = min(case["nz"], -(-_layers(case) // members))
    active = (nodes // (case["degree"] * case["nz"] + 1)) * \
        (case["degree"] * layers + 1) * members
    # per cell and evaluation: 6 one-dimensional sweeps forth and 6 back
    # (values, and a derivative along each axis) of 2 N flops per entry, and
    # about 40 flops of physics at each point
    evaluation = cells * (12 * N ** 3 * 2 * N + 40 * N ** 3)
    if kind == "vmult":
        powder = 0
        if case["material"] == "slp":
            powder = 16.0 * N ** 3 * case["nx"] * case["ny"] * 4
        return {"bytes": 8.0 * active + 8.0 * nodes + powder + cells,
                "flops": float(evaluation)}
    evals = case["n_steps"] * STAGES[case["method"]]
    if kind in ("steps", "ensemble"):
        # temperatures in and out, the lumped mass and the flags
        return {"bytes": 24.0 * active + 16.0 * (nodes * members - active)
                + cells, "flops": float(evaluation) * evals}
    # a gradient: the forward run, and its transposition on two fields
    return {"bytes": 16.0 * active + 16.0 * nodes * members,
            "flops": 3.0 * evaluation * evals}


def tolerance(case):
    """float64 sums. Against ``exact`` the outputs lie within 3e-14 (a single
    operator application) to 7e-13 (deposition steps, a point near the
    solidus) and the gradients within 2e-11; ``max`` allows that error to sit
    at a few nodes."""
    if case["kind"] in ("gradient", "gradients"):
        return {"rel": 1e-10, "max": 1e-7}
    if case["kind"] == "analysis":
        return {"rel": 1e-12, "max": 1e-9}
    return {"rel": 3e-12, "max": 1e-9}


# ---------------------------------------------------------------------------
# the same results from plain float64 torch
# ---------------------------------------------------------------------------

def _lobatto(p):
    """Gauss-Lobatto points and weights on [0, 1] for degree p."""
    L = np.polynomial.legendre.Legendre.basis(p)
    x = np.concatenate([[-1.0], np.sort(L.deriv().roots().real), [1.0]])
    w = 2.0 / (p * (p + 1) * L(x) ** 2)
    return 0.5 * (x + 1.0), 0.5 * w


def _beam_at(p, t):
    """Centre and power factor of the first beam at time t."""
    t0, a = 0.0, np.array(p.beams[0].segments[0][2], float)
    for end, power, xyz in p.beams[0].segments:
        b = np.array(xyz, float)
        if t <= end:
            return a + (b - a) * ((t - t0) / (end - t0)), power
        t0, a = end, b
    return a, 0.0


class _Model:
    """The operator of one problem (or of one member of an ensemble)."""

    def __init__(self, p, member=None):
        f64 = dict(dtype=torch.float64, device="cuda")
        member = member or Member()
        self.p, self.n = p, p.fe_degree + 1
        n, nc, nn = self.n, p.n_cells, p.n_nodes
        self.h = [p.extent[a] / nc[a] for a in range(3)]
        xl, wl = _lobatto(p.fe_degree)
        xg, wg = np.polynomial.legendre.leggauss(n)
        xg, wg = 0.5 * (xg + 1.0), 0.5 * wg
        S, D = np.ones((n, n)), np.zeros((n, n))
        for i in range(n):
            others = [k for k in range(n) if k != i]
            poly = np.polynomial.Polynomial.fromroots(xl[others])
            poly = poly / poly(xl[i])
            S[:, i], D[:, i] = poly(xg), poly.deriv()(xg)
        self.S, self.D = torch.tensor(S, **f64), torch.tensor(D, **f64)
        self.xg, w = torch.tensor(xg, **f64), torch.tensor(wg, **f64)
        det = self.h[0] * self.h[1] * self.h[2]
        self.jxw = det * w[:, None, None] * w[:, None] * w
        act = member.cell_active if member.cell_active is not None \
            else p.cell_active
        act = np.ones(p.n_cells_total, bool) if act is None else \
            np.asarray(act).astype(bool)
        cells = np.nonzero(act)[0]
        self.cc = [torch.tensor(v, device="cuda") for v in (
            cells % nc[0], (cells // nc[0]) % nc[1],
            cells // (nc[0] * nc[1]))]
        k = torch.arange(n, device="cuda")
        at = [self.cc[a][:, None] * p.fe_degree + k for a in range(3)]
        self.idx = (at[0][:, None, None, :] +
                    nn[0] * (at[1][:, None, :, None] +
                             nn[1] * at[2][:, :, None, None]))
        st = member.cell_state if member.cell_state is not None \
            else p.cell_state
        self.powder = None
        if p.material.n_states == 3:
            pw = np.zeros(p.n_cells_total) if st is None else \
                np.asarray(st).reshape(p.n_cells_total, 3)[:, 2]
            self.powder = torch.tensor(pw[cells], **f64)[
                :, None, None, None].expand(self.idx.shape)
        mass = torch.zeros(p.n_dofs, **f64)
        gl = torch.tensor(wl, **f64)
        lump = det * gl[:, None, None] * gl[:, None] * gl
        mass.index_add_(0, self.idx.reshape(-1),
                        lump.expand(self.idx.shape).reshape(-1))
        self.inv_mass = torch.where(mass > 0, 1.0 / mass, 0.0 * mass)
        # faces with a boundary term: the top of the box and the faces
        # towards inactive cells
        self.faces = []
        if p.boundary_types[-1] != 1:
            grid = torch.tensor(act.reshape(nc[2], nc[1], nc[0]),
                                device="cuda")
            x, y, z = self.cc
            for d in range(3):
                for side in (0, 1):
                    nb = [x, y, z]
                    nb[d] = nb[d] + (1 if side else -1)
                    out = (nb[d] < 0) | (nb[d] >= nc[d])
                    q = [torch.clamp(nb[a], 0, nc[a] - 1) for a in range(3)]
                    on = ~out & ~grid[q[2], q[1], q[0]]
                    if (d, side) == (2, 1):
                        on |= out
                    sel = torch.nonzero(on)[:, 0]
                    if not len(sel):
                        continue
                    ix = self.idx[sel].select(3 - d, n - 1 if side else 0)
                    area = det / self.h[d]
                    fp = None if self.powder is None else \
                        self.powder[sel].select(3 - d, 0)
                    self.faces.append((ix, area * w[:, None] * w, fp))
        m, self.k_scale = p.material, member.conductivity_scale
        self.m = m
        self.table = [[torch.tensor(m.table[0, q, s], **f64)
                       for s in range(m.n_states)] for q in range(8)]
        b = p.beams[0]
        eta = b.absorption_efficiency if member.absorption_efficiency is None \
            else member.absorption_efficiency[0]
        power = b.max_power if member.max_power is None else \
            member.max_power[0]
        self.power = power
        self.theta = torch.tensor([float(eta), 1.0, b.radius], **f64)

    def state(self):
        return [self.powder] + [f[2] for f in self.faces]

    def prop(self, k, T, r):
        """Property k of the mixture with state ratios r."""
        v = 0.0
        for s in range(self.m.n_states):
            if self.m.use_table:
                tab = self.table[k][s]
                j = torch.searchsorted(tab[:, 0].contiguous(), T.detach(),
                                       right=True)
                a, b = (j - 1).clamp(0, 11), j.clamp(0, 11)
                ta, tb, va, vb = tab[a, 0], tab[b, 0], tab[a, 1], tab[b, 1]
                same = ta == tb
                slope = torch.where(same, 0.0 * ta, (vb - va) /
                                    torch.where(same, 1.0 + 0.0 * ta, tb - ta))
                inside = (j > 0) & (j < 12)
                x = torch.where(inside, va + (T - ta) * slope, va)
            else:
                x = 0.0 * T
                for c in self.m.poly[0, k, s, :self.m.p_order + 1][::-1]:
                    x = x * T + float(c)
            v = v + r[s] * x
        return v

    def ratios(self, T, powder):
        """State ratios, 1 / (rho c_p) and the powder ratio after."""
        m = self.m
        if m.n_states == 1:
            r, latent = [torch.ones_like(T)], 0.0
        else:
            liquidus, solidus, heat = m.prop[0, 0], m.prop[0, 1], m.prop[0, 2]
            l = ((T - solidus) / (liquidus - solidus)).clamp(0.0, 1.0)
            powder = torch.where(powder < 1.0 - l, powder, 1.0 - l)
            r = [1.0 - l - powder, l, powder]
            latent = torch.where(r[1] * r[0] > 0.0,
                                 heat / (liquidus - solidus), 0.0)
        return r, 1.0 / (self.prop(0, T, r) *
                         (self.prop(1, T, r) + latent)), powder

    @staticmethod
    def along(M, v, axis):
        """M applied along an axis of v."""
        return torch.stack([sum(M[q, k] * v.select(axis, k)
                                for k in range(M.shape[1]))
                            for q in range(M.shape[0])], dim=axis)

    def rhs(self, T, t, state, theta=None):
        """A(T) at time t, and the powder ratios after the evaluation."""
        theta = self.theta if theta is None else theta
        p, S, D = self.p, self.S, self.D
        u = T[self.idx]
        ux = self.along(S, u, 3)
        uxy = self.along(S, ux, 2)
        v = self.along(S, uxy, 1)
        g = [self.along(S, self.along(S, self.along(D, u, 3), 2), 1),
             self.along(S, self.along(D, ux, 2), 1), self.along(D, uxy, 1)]
        r, irc, powder = self.ratios(v, state[0])
        new = [powder]
        ks = self.k_scale * theta[1]
        w = [-irc * ks * self.prop(2 + d, v, r) * g[d] * self.jxw /
             self.h[d] ** 2 for d in range(3)]
        q = irc * self.source(t, theta) * self.jxw
        St, Dt = S.T, D.T
        a = self.along(St, self.along(St, w[2], 3), 2)
        out = self.along(Dt, a, 1)
        a = self.along(Dt, self.along(St, w[1], 3), 2) + \
            self.along(St, self.along(Dt, w[0], 3) + self.along(St, q, 3), 2)
        out = out + self.along(St, a, 1)
        res = torch.zeros_like(T).index_add(0, self.idx.reshape(-1),
                                            out.reshape(-1))
        for (ix, jxw, _), fp in zip(self.faces, state[1:]):
            f = self.along(S, self.along(S, T[ix], 2), 1)
            r, irc, fp = self.ratios(f, fp)
            new.append(fp)
            m = self.m
            rad, conv = m.prop[0, 3], m.prop[0, 4]
            val = self.prop(7, f, r) * (f - conv) + \
                self.prop(5, f, r) * STEFAN_BOLTZMANN * (f + rad) * \
                (f * f + rad * rad) * (f - rad)
            val = self.along(St, self.along(St, -irc * val * jxw, 2), 1)
            res = res.index_add(0, ix.reshape(-1), val.reshape(-1))
        return res, new

    def source(self, t, theta):
        b = self.p.beams[0]
        c, power = _beam_at(self.p, t)
        x, y, z = ((self.cc[a][:, None] + self.xg) * self.h[a] - float(c[a])
                   for a in range(3))
        z, r2 = z[:, :, None, None], x[:, None, None, :] ** 2 + \
            y[:, None, :, None] ** 2
        eta, radius = theta[0], theta[2]
        on = (z + b.depth >= 0.0) & (5.0 * radius.detach() ** 2 - r2 >= 0.0)
        a = eta * self.power * power / (radius ** 2 * b.depth)
        if b.type == SOURCE_GOLDAK:
            v = 2.0 * a / (math.pi / 3.0) ** 1.5 * torch.exp(
                -3.0 * (z ** 2 / b.depth ** 2 + r2 / radius ** 2))
        else:
            zr, l = z / b.depth, math.log(0.1)
            v = -a * l / math.pi * torch.exp(l * r2 / radius ** 2) * (
                -3.0 * zr ** 2 - 2.0 * zr + 1.0)
        return torch.where(on, v, 0.0 * v)

    def steps(self, method, T, t, dt, n_steps, theta=None):
        state = self.state()
        a, b, c = {"fe": ([[]], [1.0], [0.0]),
                   "rk3": ([[], [0.5], [-1.0, 2.0]],
                           [1 / 6, 2 / 3, 1 / 6], [0.0, 0.5, 1.0]),
                   "rk4": ([[], [0.5], [0.0, 0.5], [0.0, 0.0, 1.0]],
                           [1 / 6, 1 / 3, 1 / 3, 1 / 6],
                           [0.0, 0.5, 0.5, 1.0])}[method]
        for _ in range(n_steps):
            f = []
            for i in range(len(b)):
                Y = T
                for k, aik in enumerate(a[i]):
                    if aik:
                        Y = Y + dt * aik * f[k]
                r, state = self.rhs(Y, t + c[i] * dt, state, theta)
                f.append(r * self.inv_mass)
            for i, bi in enumerate(b):
                T = T + dt * bi * f[i]
            t = t + dt
        return T


def _exact_gradient(model, c, T0, t, obs, y):
    T0 = T0.clone().requires_grad_(True)
    theta = model.theta.clone().requires_grad_(True)
    T = model.steps(c["method"], T0, t, c["dt"], c["n_steps"], theta)
    at = torch.tensor(obs, device="cuda")
    J = 0.5 * ((T[at] - torch.tensor(y, device="cuda")) ** 2).sum()
    lam, g = torch.autograd.grad(J, (T0, theta))
    return float(J), g.cpu().numpy(), T.detach(), lam


def _exact_analysis(c, s):
    p, X = s["problem"], s["X"]
    dev = dict(dtype=torch.float64, device="cuda")
    N, obs = X.shape[0], torch.tensor(s["obs"], device="cuda")
    A = X - X.mean(dim=0)
    S = A[:, obs]
    D = torch.tensor(s["noise"], **dev) + torch.tensor(s["y"], **dev) - \
        X[:, obs]
    xyz = _axes(p)
    nn = p.n_nodes
    every = torch.arange(p.n_dofs, device="cuda")

    def factor(nodes):
        if c["localization"] == "none":
            return 1.0
        d2 = 0.0
        for x, k in zip(xyz, (lambda i: i % nn[0], lambda i: (i // nn[0]) %
                              nn[1], lambda i: i // (nn[0] * nn[1]))):
            d2 = d2 + (x[k(nodes)][:, None] - x[k(obs)]) ** 2
        d = torch.sqrt(d2)
        rho = torch.ones_like(d)
        if c["localization"] == "gaspari_cohn":
            r = 2.0 * d / c["cutoff"]
            rho = torch.where(
                r < 1.0, 1 - 5 / 3 * r ** 2 + 5 / 8 * r ** 3 + r ** 4 / 2 -
                r ** 5 / 4, 4 - 5 * r + 5 / 3 * r ** 2 + 5 / 8 * r ** 3 -
                r ** 4 / 2 + r ** 5 / 12 - 2 / (3 * r.clamp(min=1e-9)))
        return torch.where(d <= c["cutoff"], rho, 0.0 * rho)

    C = factor(obs) * (S.T.contiguous() @ S) / (N - 1) + \
        torch.tensor(s["R"], **dev)
    E = torch.linalg.solve(C.cpu(), D.T.contiguous().cpu()).cuda()
    out = X.clone()
    for k in range(0, p.n_dofs, 65536):
        part = every[k:k + 65536]
        G = (A[:, part].T.contiguous() @ S) * factor(part) / (N - 1)
        out[:, part] += (G @ E).T
    par = torch.tensor(s["params"], **dev)
    Ap = par - par.mean(dim=0)
    par = par + ((Ap.T.contiguous() @ S) / (N - 1) @ E).T
    return {"X": out, "params": par.cpu().numpy()}


def exact(case, seed):
    s = _inputs(case, seed)
    p, kind, t = s["problem"], case["kind"], s["t"]
    if kind == "analysis":
        return _exact_analysis(case, s)
    members = s["members"] or [None]
    if kind in ("gradient", "gradients"):
        got = [_exact_gradient(_Model(p, m), case, s["T"][j], t, s["obs"],
                               s["y"][j]) for j, m in enumerate(members)]
        J, grad, T, lam = (list(v) for v in zip(*got))
        if kind == "gradient":
            return {"J": J[0], "grad": grad[0], "T_final": T[0],
                    "lambda0": lam[0]}
        return {"J": np.array(J), "grad": np.stack(grad),
                "T_final": torch.stack(T), "lambda0": torch.stack(lam)}
    with torch.no_grad():
        if kind == "vmult":
            model = _Model(p)
            return model.rhs(s["T"][0], t, model.state())[0]
        out = [_Model(p, m).steps(case["method"], s["T"][j], t, case["dt"],
                                  case["n_steps"])
               for j, m in enumerate(members)]
    return out[0] if s["members"] is None else torch.stack(out)
