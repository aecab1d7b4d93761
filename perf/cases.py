"""Performance cases of the PIC time step: what is timed, on which inputs, and
what the outputs should be in 64-bit arithmetic.

A case is a dict of plain values.  Its "kind" is the way a program drives the
library:

    driver   the loop of mandor_core: one step() with its energies per
             iteration, then the field half of a checkpoint;
    probes   the same loop with probes set: the stages one by one, a probe
             sample after the H half step;
    advance  steps enqueued without host synchronisation, then the energy
             history and the fields;
    slices   an ensemble of scan runs advanced together in slices of 25 steps,
             as the serving loop does, then every run's result;
    record   a few steps, then a full output record: checkpoint (fields and
             markers) and Tecplot payloads (node values of E, H, J and the
             charge density).

and its "plasma" the initial state: "box" (the two-stream box: every cell
filled, uniform random positions), "foil" (a scan point of the serving loop:
laser on a foil; "thickness" of many wavelengths fills the box) or
"laser-foil" (the benchmark's 256 x 128 x 128 workload).

The FP32 split form's values are handed on in FP32, the FP64 form's in FP64.
exact() is the same scheme restated in plain torch at 64 bits: Yee update with
periodic, mirror and first-order Mur walls, Boris push, charge-conserving
deposit with the trajectory cut at cell faces, J fold, VSP filter, laser plane.
"""
import math

import numpy as np
import torch

import mandor3_amd as ma
from mandor3_amd import workloads

WALLS = {"p": ma.BC_PERIODIC, "m": ma.BC_MIRROR, "o": ma.BC_OPEN}
SLICE = 25                      # steps per slice of the serving loop


def _box(n, ppc, precision, steps, kind="advance", walls="pppppp", vsp=1.0):
    return dict(kind=kind, plasma="box", nx=n[0], ny=n[1], nz=n[2], ppc=ppc, precision=precision,
                steps=steps, walls=walls, vsp=vsp)


def _foil(n, ppc, precision, steps, kind="advance", a0=2.0, density=20.0, thickness=0.5,
          graphs=True):
    return dict(kind=kind, plasma="foil", nx=n[0], ny=n[1], nz=n[2], ppc=ppc, precision=precision,
                steps=steps, a0=a0, density=density, thickness=thickness, graphs=graphs)


def listed():
    return [
        # the smallest call: a few driver steps of a tiny box, where launches, the
        # per-step read-back of the energies and synchronisation are everything
        dict(_box((12, 12, 12), 8, "fp64", 4, "driver"), name="driver box 12^3 fp64"),
        # mandor_core's own loop on the two-stream box, its default form
        dict(_box((32, 32, 32), 8, "fp64", 20, "driver"), name="driver box 32^3 fp64"),
        # a run with probes, mixed walls and the VSP filter on an odd grid
        dict(_box((45, 38, 31), 4, "fp64", 10, "probes", walls="opmopm", vsp=0.8),
             name="probes mixed walls vsp"),
        # the same two-stream box in the split form, steps enqueued ahead
        dict(_box((32, 32, 32), 8, "fp32", 50), name="advance box 32^3 fp32"),
        # ordinary scan points run alone, with graph replay as the server starts them
        dict(_foil((64, 64, 64), 8, "fp32", 50), name="foil 64^3 fp32"),
        dict(_foil((128, 64, 64), 16, "fp64", 25), name="foil 128x64x64 fp64"),
        # the benchmark's headline workload in both forms
        dict(kind="advance", plasma="laser-foil", precision="fp32", steps=50, name="laser-foil fp32"),
        dict(kind="advance", plasma="laser-foil", precision="fp64", steps=25, name="laser-foil fp64"),
        # plasma in every cell (the full-box fill), where the push is nearly all
        dict(_foil((64, 64, 64), 16, "fp32", 20, thickness=8.0, density=5.0, graphs=False),
             name="full box 64^3 fp32"),
        # the serving loop's resident set: two slices of a dozen scan runs
        dict(kind="slices", plasma="scan", runs=12, precision="fp32", name="serve 12 runs fp32"),
        dict(kind="slices", plasma="scan", runs=5, precision="fp64", name="serve 5 runs fp64"),
        # a full output record of an ordinary run
        dict(_foil((96, 48, 48), 16, "fp32", 10, "record"), name="record foil 96x48x48 fp32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["driver", "probes", "advance", "advance", "advance", "slices", "record"])
    precision = rng.choice(["fp32", "fp64"])
    if kind == "slices":
        return dict(kind="slices", plasma="scan", runs=rng.randint(2, 10 if precision == "fp32" else 5),
                    precision=precision)
    if kind in ("driver", "probes") or (kind == "advance" and rng.random() < 0.35):
        n = [_log(rng, 8, 48) for _ in range(3)]
        walls = "pppppp"
        if rng.random() < 0.6:
            ax = [rng.choice(["pp", "mm", "oo", "om", "mo"]) for _ in range(3)]
            walls = "".join(a[0] for a in ax) + "".join(a[1] for a in ax)
        vsp = rng.choice([1.0, 1.0, round(rng.uniform(0.55, 0.95), 2)])
        return _box(n, rng.choice([2, 4, 8]), precision, _log(rng, 3, 20 if kind != "advance" else 50),
                    kind, walls, vsp)
    big = rng.random() < 0.3
    n = [_log(rng, 32, 160 if big else 96)] + [_log(rng, 20, 96 if big else 64) for _ in range(2)]
    return _foil(n, rng.choice([4, 8, 16, 27, 32]), precision,
                 rng.randint(5, 15) if kind == "record" else rng.randint(10, 40), kind,
                 a0=round(math.exp(rng.uniform(math.log(0.5), math.log(4.0))), 3),
                 density=round(rng.uniform(5, 50), 2), thickness=round(rng.uniform(0.2, 1.0), 2),
                 graphs=rng.random() < 0.5)


# ---------------- initial states ----------------
def _box_state(case, seed):
    """Every cell filled with ppc electrons (vth 0.05 c, beams +-0.2 c along x)
    at uniform random positions and a cold ion where each electron sits."""
    n = (case["nx"], case["ny"], case["nz"])
    h = (0.05, 0.05, 0.05)
    rng = np.random.default_rng([seed, n[0], n[1], n[2]])
    N = n[0] * n[1] * n[2] * case["ppc"]
    c = np.arange(N) // case["ppc"]
    cells = np.stack([c // (n[1] * n[2]), c // n[2] % n[1], c % n[2]], -1)
    pos = (cells + rng.random((N, 3))) * 0.05
    u = rng.standard_normal((N, 3)) * 0.05
    u[:, 0] += np.where(np.arange(N) % 2 == 0, 0.2, -0.2)
    M = np.zeros(2 * N, dtype=ma.MARKER_DTYPE)
    w = workloads.RHO_CRIT / case["ppc"]
    for s, (q, qm) in enumerate(((-w, -1.0), (w, workloads.QM_PROTON))):
        V = M[s * N:(s + 1) * N]
        V["x"], V["y"], V["z"] = pos.T
        if s == 0:
            V["vx"], V["vy"], V["vz"] = u.T
        V["rho"], V["qDivM"] = q, qm
    M["id"] = np.arange(1, 2 * N + 1)
    return dict(n=n, h=h, L=tuple(a * 0.05 for a in n), tau=workloads.courant_tau(h),
                bc=tuple(WALLS[w] for w in case["walls"]), markers=M, laser=None)


def _states(case, seed):
    """The initial state of every run of a case."""
    if case["plasma"] == "box":
        return [_box_state(case, seed)]
    if case["plasma"] == "laser-foil":
        return [workloads.laser_foil(seed=seed)]
    if case["plasma"] == "foil":
        return [workloads.foil_request((case["nx"], case["ny"], case["nz"]), case["ppc"], case["a0"],
                                       case["density"], case["thickness"], seed=seed)]
    # the scan's own draws; the set of grids is the case's, the runs' states the seed's
    rng = np.random.default_rng(1000 + case["runs"])
    out = []
    for q in range(case["runs"]):
        p = workloads.scan_request(rng)
        p.update(seed=seed * 64 + q)
        p.pop("steps")
        out.append(workloads.foil_request(**p))
    return out


def _probe_nodes(n):
    """A line along x and a rectangle across it, as run_probes.cfg lists them."""
    line = [(i, n[1] // 2, n[2] // 2) for i in range(n[0])]
    rect = [(n[0] // 2, j, k) for j in range(0, n[1], 2) for k in range(0, n[2], 2)]
    return np.array(line + rect, dtype=np.int32)


def prepare(case, seed):
    runs = []
    for st in _states(case, seed):
        r = ma.Run(st["n"], st["h"], st["L"], st["tau"], st["bc"], 0.0,
                   precision=ma.FP64 if case["precision"] == "fp64" else ma.FP32_SPLIT,
                   max_markers=max(int(st["markers"].size), 1))
        z = np.zeros(3 * r.nodes)
        r.set_fields(z, z)
        r.load_markers(st["markers"])
        if st["laser"] is not None:
            r.add_laser(*st["laser"])
        if case.get("vsp", 1.0) != 1.0:
            r.set_vsp(case["vsp"])
        r.init()
        if case["kind"] == "slices" or case.get("graphs"):
            r.set_graphs(True)
        if case["kind"] == "probes":
            r.set_probes(_probe_nodes(st["n"]))
        runs.append(r)
    return dict(case=case, runs=runs, loaded=int(st["markers"].size))


# ---------------- one pass ----------------
def _as_form(case, a):
    """The FP64 form's values as they are, the split form's in FP32."""
    t = torch.from_numpy(np.ascontiguousarray(a))
    return t if case["precision"] == "fp64" else t.float()


def _fields(case, r):
    E, H = r.fields()
    return {"E": _as_form(case, E), "H": _as_form(case, H)}


def _by_id(case, M, n):
    """Marker positions and momenta in the order of the tracer ids."""
    out = np.zeros((n, 6))
    at = M["id"] - 1
    for c, f in enumerate(("x", "y", "z", "vx", "vy", "vz")):
        out[at, c] = M[f]
    return _as_form(case, out)


def run(state):
    case, runs = state["case"], state["runs"]
    r = runs[0]
    if case["kind"] == "driver":
        diag = np.stack([r.step(diag=True) for _ in range(case["steps"])])
        return dict(_fields(case, r), diag=_as_form(case, diag))
    if case["kind"] == "probes":
        diag, samples = [], []
        for _ in range(case["steps"]):
            t = r.time
            r.stage("em_h_half")
            we, wm = r.energy()
            samples.append(r.probe_sample())
            r.stage("push_deposit")
            wt = r.temperature()
            r.stage("em_h_step")
            r.stage("em_e_start")
            r.stage("j_finish")
            r.stage("em_e_finish")
            diag.append((t, we, wm, wt[0], wt[1], wt[2]))
        return dict(_fields(case, r), diag=_as_form(case, np.array(diag)),
                    probes=_as_form(case, np.stack(samples)))
    if case["kind"] == "slices":
        for _ in range(2):
            ma.batch_advance(runs, SLICE)
            r.sync()
        return [dict(_fields(case, q), diag=_as_form(case, q.diag_history(2 * SLICE))) for q in runs]
    r.advance(case["steps"])
    out = dict(diag=_as_form(case, r.diag_history(case["steps"])))
    out.update(_fields(case, r))
    if case["kind"] == "record":
        for what, name in enumerate(("nodeE", "nodeH", "nodeJ")):
            out[name] = _as_form(case, r.node_fields(what))
        out["rho"] = _as_form(case, r.rho())
        out["markers"] = _by_id(case, r.markers(), state["loaded"])
    return out


# ---------------- what a pass cannot do without ----------------
def _sizes(case):
    """(cells, markers) of every run."""
    if case["plasma"] == "box":
        return [((case["nx"], case["ny"], case["nz"]),
                 2 * case["ppc"] * case["nx"] * case["ny"] * case["nz"])]
    if case["plasma"] == "laser-foil":
        return [((256, 128, 128), 8573040)]

    def foil(n, ppc, thickness):
        xc, half = int(round(0.625 * n[0])), max(1, int(round(thickness / 0.05 / 2)))
        i0, i1 = max(xc - half, 8), min(xc + half, n[0] - 3)
        return tuple(n), 2 * ppc * (i1 - i0) * (n[1] - 4) * (n[2] - 4)

    if case["plasma"] == "foil":
        return [foil((case["nx"], case["ny"], case["nz"]), case["ppc"], case["thickness"])]
    rng = np.random.default_rng(1000 + case["runs"])
    out = []
    for _ in range(case["runs"]):
        p = workloads.scan_request(rng)
        out.append(foil(p["n"], p["ppc"], p["thickness"]))
    return out


def work(case):
    """Per step every marker's state and id and every node's E and H are read
    and written once; the results are written once as they leave."""
    wide = case["precision"] == "fp64"
    steps = 2 * SLICE if case["kind"] == "slices" else case["steps"]
    nbytes = flops = 0
    for n, markers in _sizes(case):
        nodes = (n[0] + 1) * (n[1] + 1) * (n[2] + 1)
        nbytes += steps * (markers * 2 * (60 if wide else 36) + nodes * 2 * 6 * (8 if wide else 4))
        nbytes += nodes * 6 * 8
        flops += steps * (markers * 400 + nodes * 36)
        if case["kind"] == "record":
            nbytes += nodes * (9 + 1) * 8 + markers * 48
        if case["kind"] == "probes":
            nbytes += steps * len(_probe_nodes(n)) * 48
    return {"bytes": nbytes, "flops": flops}


# ---------------- the scheme in 64 bits ----------------
class _Exact:
    """One run in plain torch float64; arrays cover the nodes [-2, n+2]."""

    def __init__(self, st, vsp):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.n, self.h, self.tau, self.bc, self.vsp = st["n"], st["h"], st["tau"], st["bc"], vsp
        self.L = [a * b for a, b in zip(st["n"], st["h"])]
        self.shape = tuple(a + 5 for a in self.n)
        self.E, self.H = self._mesh(3), self._mesh(3)
        self.mur = {}
        self.time = 0.0
        M = st["markers"]
        col = lambda *f: torch.from_numpy(np.stack([M[c].astype(np.float64) for c in f])).to(self.dev)
        self.x, self.u = col("x", "y", "z"), col("vx", "vy", "vz")
        self.w, self.qm, self.id = col("rho")[0], col("qDivM")[0], col("id")[0].long()
        self._marker_walls()
        self.laser = None
        if st["laser"] is not None:
            p, m = st["laser"]
            self.laser = p, torch.from_numpy(m).to(self.dev).reshape(2, self.n[1] - 9, self.n[2] - 9, 4)

    def _mesh(self, c):
        return torch.zeros((c,) + self.shape, dtype=torch.float64, device=self.dev)

    def _at(self, F, ea, a):
        """The layer of nodes a of axis ea, transverse nodes [0, n+1]."""
        s = [slice(2, v + 4) for v in self.n]
        s[ea] = a + 2
        return F[tuple(s)]

    def _walls(self, X, electric):
        for ea in range(3):
            ep, eq, N = (ea + 1) % 3, (ea + 2) % 3, self.n[ea]
            for top in range(2):
                b = self.bc[3 * top + ea]
                if b == ma.BC_PERIODIC:
                    if top:
                        continue
                    for F in X:
                        v0, v1, vN = (self._at(F, ea, a).clone() for a in (0, 1, N))
                        if electric:
                            self._at(F, ea, N)[:] = v0
                        else:
                            self._at(F, ea, 0)[:] = vN
                        self._at(F, ea, N + 1)[:] = v1
                    continue
                pl = N * top
                inn, ext, nxt = pl + 1 - top, pl + top, pl + 1 - 2 * top
                if not electric:
                    if b == ma.BC_MIRROR:
                        self._at(X[ea], ea, pl)[:] = 0
                    for c in (ep, eq):
                        self._at(X[c], ea, ext)[:] = self._at(X[c], ea, inn).clone()
                    continue
                normal = self._at(X[ea], ea, inn).clone()
                for c in (ep, eq):
                    if b == ma.BC_MIRROR:
                        self._at(X[c], ea, pl)[:] = 0
                        continue
                    near = self._at(X[c], ea, nxt).clone()
                    old = self.mur.get((ea, top, c), (torch.zeros_like(near), torch.zeros_like(near)))
                    alpha = (self.tau - self.h[ea]) / (self.tau + self.h[ea])
                    plane = old[1] + alpha * (near - old[0])
                    self._at(X[c], ea, pl)[:] = plane
                    self.mur[ea, top, c] = plane, near
                self._at(X[ea], ea, ext)[:] = normal

    def _curl(self, F, sign):
        """curl of F from differences towards lower (sign -1) or higher nodes."""
        def d(c, ax):
            s = torch.roll(F[c], -sign, ax)
            return (s - F[c]) * sign / self.h[ax]
        return torch.stack([d(2, 1) - d(1, 2), d(0, 2) - d(2, 0), d(1, 0) - d(0, 1)])

    def _update(self, X, dX, electric):
        """X + dX on the nodes the Yee scheme advances, then the walls."""
        out = X.clone()
        s = [slice(None)]
        for a in range(3):
            lo = {ma.BC_PERIODIC: 0, ma.BC_MIRROR: 1, ma.BC_OPEN: int(electric)}[self.bc[a]]
            hi = self.n[a] - (1 if electric and self.bc[3 + a] == ma.BC_PERIODIC else 0)
            s.append(slice(lo + 2, hi + 3))
        out[tuple(s)] += dX[tuple(s)]
        self._walls(out, electric)
        return out

    def _laser_plane(self, F, electric):
        if self.laser is None:
            return
        (A, T0, delay, dt, phi0, _, plane), m = self.laser
        t = self.time + (0.5 * self.tau if electric else 0.0) - T0 + delay
        amp = math.exp(-(2 * t / dt) ** 2) * self.tau / self.h[0]
        cs, sn = math.cos(2 * math.pi * t + phi0), math.sin(2 * math.pi * t + phi0)
        m = m[1 if electric else 0]
        lo, hi = ([5] * 2, [v - 5 for v in self.n[1:]])
        s = (plane - (1 if electric else 0) + 2, slice(lo[0] + 2, hi[0] + 3), slice(lo[1] + 2, hi[1] + 3))
        F[1][s] += amp * (m[..., 2] * cs + m[..., 3] * sn)
        F[2][s] += amp * (m[..., 0] * cs + m[..., 1] * sn)

    def _flat(self, i, j, k):
        return ((i + 2) * self.shape[1] + (j + 2)) * self.shape[2] + (k + 2)

    def _gather(self, F, cell, frac):
        f, base = F.reshape(-1), self._flat(*cell)
        out = 0
        for a in range(8):
            d = (a >> 2, a >> 1 & 1, a & 1)
            wt = 1.0
            for q in range(3):
                wt = wt * (frac[q] if d[q] else 1 - frac[q])
            out = out + wt * f[base + (d[0] * self.shape[1] + d[1]) * self.shape[2] + d[2]]
        return out

    def _deposit(self, J, cell, r1, r2, w):
        """One straight segment inside its cell; r1, r2 in cell units from it."""
        d, m = r2 - r1, 0.5 * (r1 + r2)
        flat = [J[c].reshape(-1) for c in range(3)]
        base = self._flat(*cell)
        step = (self.shape[1] * self.shape[2], self.shape[2], 1)
        for c in range(3):
            p, q = [a for a in range(3) if a != c]
            cur = w * d[c] * self.h[c] / self.tau
            cross = d[p] * d[q] / 12
            for a in range(4):
                up, uq = a & 1, a >> 1
                v = (m[p] if up else 1 - m[p]) * (m[q] if uq else 1 - m[q])
                v = cur * (v + (cross if up == uq else -cross))
                flat[c].index_add_(0, base + step[c] + up * step[p] + uq * step[q], v)

    def _marker_walls(self):
        live = torch.ones_like(self.w, dtype=torch.bool)
        for top in range(2):
            for a in range(3):
                b, x = self.bc[3 * top + a], self.x[a]
                lim = self.L[a] if top else 0.0
                if b == ma.BC_OPEN:
                    live &= (x < lim - self.h[a]) if top else (x > self.h[a])
                    continue
                out = (x >= lim) if top else (x <= lim)
                if b == ma.BC_PERIODIC:
                    x += out.double() * (-self.L[a] if top else self.L[a])
                else:
                    self.x[a] = torch.where(out, 2 * lim - x, x)
                    self.u[a] = torch.where(out, -self.u[a], self.u[a])
        if not bool(live.all()):
            self.x, self.u = self.x[:, live], self.u[:, live]
            self.w, self.qm, self.id = self.w[live], self.qm[live], self.id[live]

    def _push(self, E, H):
        g = [self.x[a] / self.h[a] for a in range(3)]
        cell = [torch.floor(v).long() for v in g]
        frac = [v - c for v, c in zip(g, cell)]
        half = [torch.floor(v + 0.5).long() for v in g]
        hfrac = [v + 0.5 - c for v, c in zip(g, half)]
        pick = lambda m: ([half[a] if m[a] else cell[a] for a in range(3)],
                          [hfrac[a] if m[a] else frac[a] for a in range(3)])
        e = [self._gather(E[c], *pick([a == c for a in range(3)])) for c in range(3)]
        b = [self._gather(H[c], *pick([a != c for a in range(3)])) for c in range(3)]
        tm = 0.5 * self.tau * self.qm
        p = torch.stack([self.u[c] + tm * e[c] for c in range(3)])
        p2 = (p * p).sum(0)
        gam = torch.sqrt(1 + p2)
        vol = self.h[0] * self.h[1] * self.h[2]
        wt = (gam - 1) * self.w / (p2 + 1e-19) * vol / self.qm
        self.wt = [float((wt * p[c] * p[c]).sum()) for c in range(3)]
        t = torch.stack([tm / gam * b[c] for c in range(3)])
        cross = lambda a, c: torch.stack([a[1] * c[2] - a[2] * c[1], a[2] * c[0] - a[0] * c[2],
                                          a[0] * c[1] - a[1] * c[0]])
        v = p + cross(p, t)
        v = p + cross(v, t * (2 / (1 + (t * t).sum(0))))
        self.u = v + torch.stack([tm * e[c] for c in range(3)])
        dx = self.u * (self.tau / torch.sqrt(1 + (self.u * self.u).sum(0)))
        # the move in cell units from the start cell, cut where it crosses a face
        r1 = torch.stack(frac)
        r2 = torch.stack([frac[a] + dx[a] / self.h[a] for a in range(3)])
        to = torch.floor(r2).long()
        at = torch.where(to != 0, ((to > 0).double() - r1) / torch.where(to != 0, r2 - r1, 1.0), 2.0)
        J = self._mesh(3)
        order = torch.argsort(at, 0)
        cuts = torch.gather(at, 0, order).clamp(max=1.0)
        here = torch.stack(cell)
        start, last, sel = here.clone(), torch.zeros_like(cuts[0]), slice(None)
        for s in range(4):
            nxt = cuts[s] if s < 3 else torch.ones_like(last)
            if s:
                sel = (at.gather(0, order[s - 1:s])[0] <= 1.0).nonzero()[:, 0]
                if sel.numel() == 0:
                    break
                ax = order[s - 1][sel]
                here[ax, sel] += to[ax, sel]
            o = (here - start)[:, sel]
            q1 = r1[:, sel] + last[sel] * (r2 - r1)[:, sel] - o
            q2 = r1[:, sel] + nxt[sel] * (r2 - r1)[:, sel] - o
            self._deposit(J, [here[a][sel] for a in range(3)], q1, q2, self.w[sel])
            last = nxt
        self.x = self.x + dx
        self._marker_walls()
        return J

    def _fold(self, F, current):
        """J (three components) or rho (one) folded at the walls."""
        at = lambda f, ea, a: f.select(ea, a + 2)
        for ea in range(3):
            N, tang = self.n[ea], [c for c in range(3) if c != ea] if current else [0]
            if self.bc[ea] == ma.BC_PERIODIC:
                for f in F:
                    for a in range(-2, 3):
                        v = at(f, ea, a) + at(f, ea, a + N)
                        at(f, ea, a)[:] = v
                        at(f, ea, a + N)[:] = v
                continue
            for top in range(2):
                pl, so = N * top, 2 * top - 1
                if current:
                    inn, ext = pl + 1 - top, pl + top
                    for s in range(2):
                        v = at(F[ea], ea, inn - s * so) - at(F[ea], ea, ext + s * so)
                        at(F[ea], ea, inn - s * so)[:] = v
                        at(F[ea], ea, ext + s * so)[:] = v
                for c in tang:
                    for s in (1, 2):
                        v = at(F[c], ea, pl - s * so) + at(F[c], ea, pl + s * so)
                        at(F[c], ea, pl - s * so)[:] = v
                        at(F[c], ea, pl + s * so)[:] = -v
                    at(F[c], ea, pl)[:] = 0

    def _filter(self, F):
        if self.vsp == 1.0:
            return
        beta = 0.5 * (1 - self.vsp)
        for ax in (2, 1, 0):
            for f in F:
                v, n = f.clone(), f.shape[ax]
                f *= self.vsp
                f.narrow(ax, 1, n - 1).add_(beta * v.narrow(ax, 0, n - 1))
                f.narrow(ax, 0, n - 1).add_(beta * v.narrow(ax, 1, n - 1))

    def rho(self):
        F = self._mesh(1)
        g = [self.x[a] / self.h[a] for a in range(3)]
        cell = [torch.floor(v).long() for v in g]
        frac = [v - c for v, c in zip(g, cell)]
        for a in range(8):
            d = (a >> 2, a >> 1 & 1, a & 1)
            wt = self.w
            for q in range(3):
                wt = wt * (frac[q] if d[q] else 1 - frac[q])
            F[0].reshape(-1).index_add_(0, self._flat(*[cell[q] + d[q] for q in range(3)]), wt)
        self._fold(F, False)
        self._filter(F)
        return F[0].reshape(-1)

    def nodes(self, what):
        F = (self.E, self.H, self.J)[what]
        n = self.n
        s = lambda f, d: f[tuple(slice(2 + d[a], n[a] + 3 + d[a]) for a in range(3))]
        unit = lambda *ax: tuple(int(a in ax) for a in range(3))
        out = []
        for c in range(3):
            if what == 1:
                p, q = [a for a in range(3) if a != c]
                out.append(0.25 * (s(F[c], unit()) + s(F[c], unit(p)) + s(F[c], unit(q)) +
                                   s(F[c], unit(p, q))))
            else:
                out.append(0.5 * (s(F[c], unit()) + s(F[c], unit(c))))
        return torch.stack(out, -1).reshape(-1, 3)

    def step(self):
        """One step; returns the energy row, leaves the fields of the half
        step (where probes sample) in self.half."""
        H1 = self._update(self.H, -self.tau * self._curl(self.E, -1), False)
        Hn = 0.5 * (self.H + H1)
        n = self.n
        s = lambda f, *ax: f[tuple(slice(2 + int(a in ax), n[a] + 2 + int(a in ax)) for a in range(3))]
        we = sum(float((s(self.E[c], c) ** 2).sum()) for c in range(3))
        wm = sum(float((s(Hn[c], *[a for a in range(3) if a != c]) ** 2).sum()) for c in range(3))
        vol = 0.5 * self.h[0] * self.h[1] * self.h[2]
        self.half = self.E, Hn
        J = self._push(self.E, Hn)
        self._laser_plane(H1, False)
        self.H = H1
        E1 = self._update(self.E, self.tau * self._curl(H1, 1), True)
        self._laser_plane(E1, True)
        self._fold(J, True)
        self._filter(J)
        self.J = J
        self.E = E1 - self.tau * J
        row = (self.time, vol * we, vol * wm) + tuple(self.wt)
        self.time += self.tau
        return row

    def fields(self):
        s = (slice(None),) + tuple(slice(2, v + 3) for v in self.n)
        return {c: F[s].permute(1, 2, 3, 0).reshape(-1).cpu() for c, F in (("E", self.E), ("H", self.H))}

    def probes(self, ijk):
        E, H = self.E, self.H
        self.E, self.H = self.half
        shape = [v + 1 for v in self.n]
        at = torch.from_numpy(np.ravel_multi_index(tuple(ijk.T.astype(np.int64)), shape)).to(self.dev)
        v = torch.cat([self.nodes(0)[at], self.nodes(1)[at]], 1).cpu()
        self.E, self.H = E, H
        return v


def exact(case, seed):
    steps = 2 * SLICE if case["kind"] == "slices" else case["steps"]
    if not torch.cuda.is_available() and sum(m for _, m in _sizes(case)) * steps > 4e6:
        return None                                  # minutes on a CPU
    out = []
    for st in _states(case, seed):
        x = _Exact(st, case.get("vsp", 1.0))
        diag, samples = [], []
        for _ in range(steps):
            diag.append(x.step())
            if case["kind"] == "probes":
                samples.append(x.probes(_probe_nodes(x.n)))
        one = dict(x.fields(), diag=torch.tensor(diag, dtype=torch.float64))
        if samples:
            one["probes"] = torch.stack(samples)
        if case["kind"] == "record":
            for what, name in enumerate(("nodeE", "nodeH", "nodeJ")):
                one[name] = x.nodes(what).cpu()
            one["rho"] = x.rho().cpu()
            m = torch.zeros((st["markers"].size, 6), dtype=torch.float64, device=x.dev)
            m[x.id - 1] = torch.cat([x.x, x.u]).T
            one["markers"] = m.cpu()
        out.append(one)
    return out if case["kind"] == "slices" else out[0]
