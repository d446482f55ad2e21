"""Performance cases of the time-stepping framework: the calls its users make, at the sizes
they make them.

`listed()` holds the named cases, `draw(rng)` gives further ones of the same ranges.  A case
is a dict of plain values:

  kind      "solver" (Solver.step), "frames" (Solver.run over moving frames), "ensemble"
            (Ensemble.step) or "train" (ground.Network.train)
  scheme    "fb" (the reference's FB_p_v step) or "rk4"
  bits      precision of the state, 64 (the default of the framework) or 32
  nx ny nz  air points; pml absorbing points per absorbing face; pore porous points (0: none)
  hills     Gaussian hills of a terrain-following grid (0: flat)
  wind      logarithmic wind (RK4 only)
  poles     poles of the ground impedance (0: none)
  tdbc      1: the East face is the recursive-convolution impedance boundary
  graph     the solver replays captured steps (use_graph)
  receivers receivers of the run; steps time steps of one pass
  state     1: the pass also fetches the fields (a run that stores or couples them)

`prepare` builds the solver a program keeps: seeded source, ground, hills and wind, and a
state in the middle of a run (smooth waves in all fields, set with set_state).  One pass
advances it by `steps` steps and returns the receiver series, as a program that records them
does.  An FP32 run's series and fields hold FP32 values (the interface widens them), and are
returned as such.  `exact` is the same time step in plain 64-bit torch.
"""
import importlib
import math

import numpy as np
import torch

C0, RHO0, GAMMA = 343.0, 1.21, 1.4
SPACING, CFL = 0.04, 0.5
ALPHA, RESIST = 2.0, 1000.0  # absorbing-layer profile
# poles and residues of the East impedance boundary (calculation_2D.h:73-75)
TD_A = (8.226223820e-01, 3.732304064e-01, 9.106232372e-02, 4.819445335e-02, 4.225250937e-01, 1.837970986e-01)
TD_R = (8.681310138e-01, 1.953722814e-01, 1.108067950e-02, 2.566498621e-03, 1.457297589e-04, 4.648583789e-02)


def _case(name, kind, scheme, bits, shape, steps, pml=20, pore=0, hills=0, wind=0, poles=0, tdbc=0, graph=0,
          receivers=32, state=0, **more):
    c = dict(kind=kind, scheme=scheme, bits=bits, nx=shape[0], ny=shape[1], nz=shape[2], steps=steps, pml=pml,
             pore=pore, hills=hills, wind=wind, poles=poles, tdbc=tdbc, graph=graph, receivers=receivers, state=state)
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the reflection column of the learned ground's training data: hundreds of short runs
        # of a 6 x 6 column over each ground's porous layer, the smallest grid in use
        _case("column_fb64", "solver", "fb", 64, (6, 6, 640), 256, pore=10, graph=1, receivers=1, walls=1),
        # the 96 x 64 x 48 benchmark grid with the reference's scheme and precision, fields fetched
        _case("small_fb64", "solver", "fb", 64, (96, 64, 48), 100, pore=8, receivers=5, state=1),
        # a ragged small domain with every RK4 extension on, fields fetched
        _case("odd_rk64", "solver", "rk4", 64, (137, 91, 53), 40, pml=10, pore=7, hills=2, wind=1, receivers=16, state=1),
        # a whole run over moving frames (the pulse is followed along y), RK4 FP32
        _case("frames_rk32", "frames", "rk4", 32, (160, 96, 64), 180, pml=12, pore=8, hills=2, wind=1, receivers=32,
              shift=16),
        # the deck shipped with the reference: 141 x 201 x 441, East impedance boundary, FP64
        _case("shipped_fb64", "solver", "fb", 64, (141, 201, 441), 20, pml=41, tdbc=1, receivers=64),
        # the 512 x 256 x 128 benchmark grid: the reference's scheme in FP32
        _case("grid_fb32", "solver", "fb", 32, (512, 256, 128), 20, pore=16, receivers=512),
        # the same grid with the benchmark's integrator, terrain and wind, FP32 and FP64
        _case("grid_rk32", "solver", "rk4", 32, (512, 256, 128), 8, pore=16, hills=1, wind=1, receivers=512),
        _case("grid_rk64", "solver", "rk4", 64, (512, 256, 128), 6, pore=16, hills=1, wind=1, receivers=512),
        # the precision study's grid over six hills without wind, the largest domain
        _case("large_rk32", "solver", "rk4", 32, (768, 384, 192), 4, pore=24, hills=6, receivers=512),
        # the parameter sweep: uneven domains over grounds of their own, stepped together
        _case("sweep_rk32", "ensemble", "rk4", 32, (128, 96, 64), 16, pml=10, pore=16, wind=1, graph=1, receivers=4,
              members=32),
        # the learned ground in use: the impedance closure under air over a hill, FP32
        _case("closure_fb32", "solver", "fb", 32, (640, 320, 144), 12, hills=1, poles=8, receivers=512),
        # training of the ground network: shuffled batches of 32 over a few hundred grounds
        dict(name="train_net", kind="train", rows=256, batch=32, epochs=10),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.08:
        return dict(kind="train", rows=_log(rng, 48, 400), batch=rng.choice((16, 32, 64)), epochs=rng.randint(4, 10))
    if rng.random() < 0.12:
        return _case("", "ensemble", "rk4", rng.choice((32, 32, 64)), (rng.randint(90, 128), rng.randint(64, 96), 64),
                     rng.randint(6, 16), pml=10, pore=rng.randint(6, 16), wind=rng.randint(0, 1), graph=rng.randint(0, 1),
                     receivers=4, members=_log(rng, 4, 32))
    scheme = rng.choice(("fb", "rk4"))
    bits = rng.choice((32, 64))
    nx, ny, nz = _log(rng, 40, 640), _log(rng, 40, 320), _log(rng, 36, 192)
    pml = rng.randint(6, max(7, min(20, min(nx, ny, nz) // 3)))
    steps = max(3, min(80, int(1.6e8 / (nx * ny * nz))))
    rk = scheme == "rk4"
    poles = rng.choice((0, 0, 3, 8)) if not rk else 0
    hills = rng.choice((0, 1, 2))
    return _case("", "solver", scheme, bits, (nx, ny, nz), max(3, steps // (3 if rk else 1)), pml=pml,
                 pore=0 if poles else rng.choice((0, 6, 9, 16)), hills=hills, wind=rng.randint(0, 1) if rk else 0,
                 poles=poles, graph=rng.choice((0, 0, 1)), receivers=rng.randint(4, 256),
                 state=1 if nx * ny * nz < 500000 and bits == 64 else 0)


# ------------------------------------------------------------------ inputs
def _ground(rng):
    """Flow resistivity log-uniform, porosity and tortuosity uniform, as in the sweeps."""
    return dict(sigma=float(10 ** rng.uniform(5.0, 6.3)), porosity=float(rng.uniform(0.2, 0.5)),
                tort=float(rng.uniform(1.5, 4.0)))


def _inputs(case, seed, member=0):
    """Everything the deck of a case (or of one member of a sweep) is made of, as plain values."""
    rng = np.random.default_rng([int(seed), member])
    p = dict(case)
    if case["kind"] == "ensemble":
        p["nx"] = int(rng.integers(case["nx"] // 2, case["nx"] + 1))
        p["ny"] = int(rng.integers(case["ny"] // 2, case["ny"] + 1))
        p["nz"] = int(rng.integers(3 * case["nz"] // 4, case["nz"] + 1))
        p["pore"] = int(rng.integers(4, case["pore"] + 1))
    if case["tdbc"]:
        p.update(d=0.005, c=340.0, Pav=1.0e5, dt=4e-6)
    else:
        p.update(d=SPACING, c=C0, Pav=RHO0 * C0 * C0 / GAMMA, dt=CFL * SPACING / C0)
    nx, ny, nz, d = p["nx"], p["ny"], p["nz"], p["d"]
    frames = case["kind"] == "frames"
    ytot = ny + 4 * case["shift"] if frames else ny
    p["bc"] = ((2, 3 if p["pore"] else 1, 1, 1, 1, 1) if case.get("walls") else
               (2, 3 if p["pore"] else 1, 5 if case["tdbc"] else 2, 2, 2, 2))  # N S E W F B
    p.update(_ground(rng))
    p["x0"] = -0.5 * (nx - 1) * d
    D = (nz - 1) * d
    p["hill"] = [(float(rng.uniform(0.3, 0.7) * (nx - 1) * d + p["x0"]), float(rng.uniform(0.3, 0.7) * (ytot - 1) * d),
                  float(rng.uniform(0.06, 0.14) * D / max(1, case["hills"] - 1)),
                  float(rng.uniform(0.25, 0.4) * min(nx, ny) * d + 0.3 * D)) for _ in range(case["hills"])]
    p["ustar"] = float(rng.uniform(0.2, 0.5)) if case["wind"] else 0.0
    p["src"] = (float(rng.uniform(0.4, 0.6) * (nx - 1) * d + p["x0"]), float(rng.uniform(0.3, 0.6) * (ny - 1) * d),
                float(rng.uniform(0.2, 0.5) * D))
    p["width"] = 6 * d
    r = case["poles"]
    rate = np.concatenate([[0.0], np.logspace(-2.5, 2.0, r - 1)]) if r > 1 else np.zeros(r)
    p["pole"] = [(float(a), float(q)) for a, q in zip(rng.uniform(0.05, 0.6, r), rate)]
    p["zinf"] = RHO0 * C0 * math.sqrt(p["tort"]) / p["porosity"]
    p["tau"] = p["tort"] * RHO0 / p["porosity"] / p["sigma"]
    n = case["receivers"]
    p["rec"] = np.stack([rng.integers(1, nx - 1, n), rng.integers(1, ytot - 1, n), rng.integers(1, nz - 1, n)], axis=1)
    # waves that vanish on the faces, eight points or more per wavelength, one product per field
    p["modes"] = [[int(rng.integers(1, max(2, m // 8))) for m in (nz, ny, nx)] for _ in range(4)]
    p["amp"] = [float(s * rng.uniform(0.5, 1.0)) for s in (1 / (RHO0 * C0),) * 3 + (1.0,)]
    return p


def _waves(p):
    out = []
    for (a, b, c), amp in zip(p["modes"], p["amp"]):
        fz, fy, fx = (np.sin(np.pi * m * np.arange(n) / (n - 1)) for m, n in ((a, p["nz"]), (b, p["ny"]), (c, p["nx"])))
        out.append((amp * fz)[:, None, None] * (fy[:, None] * fx[None, :])[None])
    return out


def _deck(lee, p):
    frames = p["kind"] == "frames"
    kw = dict(time_domain=p["steps"] if frames else 1 << 20)
    if frames:
        kw.update(mf_judge=1, mf_jmax=p["ny"], mf_lead_dj=p["shift"] + 1, mf_trail_dj=p["shift"] + 1, mf_ratio=0.4,
                  ijkmax=p["ny"] + 4 * p["shift"])
    d = lee.deck.box(p["nx"], p["ny"], p["nz"], p["d"], pml=p["pml"], bc=p["bc"], dt=p["dt"], c=p["c"], x0=p["x0"],
                     porous_cells=p["pore"] + 2 if p["pore"] else 0, src=p["src"], gauss_width=p["width"], pml_y_time=0,
                     gamma=GAMMA, Pav=p["Pav"], **kw)
    d.pore_q, d.pore_porosity, d.pore_resistivity = math.sqrt(p["tort"]), p["porosity"], p["sigma"]
    d.integrator = 1 if p["scheme"] == "rk4" else 0
    d.hills = list(p["hill"])
    if p["wind"]:
        d.velocity_method, d.wind_ustar, d.wind_z0 = 7, p["ustar"], 0.02
    if p["poles"]:
        d.ground_poles, d.ground_zinf, d.ground_tau = p["pole"], p["zinf"], p["tau"]
    return d


def _positions(p):
    i, j, k = p["rec"].T
    d = p["d"]
    return np.stack([p["x0"] + d * i, d * j, d * k], axis=1)


def _training(case, seed):
    """Normalised grounds and smooth targets of the size of the residues' square roots."""
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1, 1, (case["rows"], 4)).astype(np.float32)
    w = rng.normal(size=(4, 8))
    t = (0.5 + 0.4 * np.tanh(x @ w + 0.3 * np.sin(3 * x[:, :1]))).astype(np.float32)
    w0 = []
    for o, i, fo, fi in ((64, 16, 64, 4), (64, 64, 64, 64), (64, 64, 64, 64), (16, 64, 8, 64)):
        W = np.zeros((o, i))
        W[:fo, :fi] = rng.uniform(-1, 1, (fo, fi)) * math.sqrt(3.0 / fi) * (0.1 if o == 16 else 1.0)
        w0 += [W.ravel(), np.zeros(o)]
    return x, t, np.concatenate(w0).astype(np.float32)


# ------------------------------------------------------------------ the cases
def prepare(case, seed):
    lee = importlib.import_module("3d_mpi_test_amd")
    if case["kind"] == "train":
        x, t, w = _training(case, seed)
        net = lee.ground.Network(seed=1)
        net.set_params(w)
        return dict(case=case, net=net, x=x, t=t)
    if case["kind"] == "ensemble":
        ps = [_inputs(case, seed, m) for m in range(case["members"])]
        e = lee.Ensemble([_deck(lee, p) for p in ps], precision=case["bits"], receivers=[_positions(p) for p in ps],
                         use_graph=bool(case["graph"]))
        for m, p in zip(e.members, ps):
            m.set_state(*_waves(p))
        return dict(case=case, ens=e)
    p = _inputs(case, seed)
    s = lee.Solver(_deck(lee, p), precision=case["bits"], receivers=_positions(p), use_graph=bool(case["graph"]))
    s.frame_setup(0)
    s.set_state(*_waves(p))
    return dict(case=case, solver=s)


def run(state):
    case = state["case"]
    if case["kind"] == "train":
        mse = state["net"].train(state["x"], state["t"], batch=case["batch"], epochs=case["epochs"], lr=2e-3, seed=7)
        return {"params": state["net"].params(), "mse": np.float32(mse)}
    kind = np.float32 if case["bits"] == 32 else np.float64
    if case["kind"] == "ensemble":
        return {"series": np.concatenate(state["ens"].step(case["steps"]), axis=1).astype(kind, copy=False)}
    s = state["solver"]
    series = s.run() if case["kind"] == "frames" else s.step(case["steps"])
    out = {"series": series.astype(kind, copy=False)}
    if case["state"]:
        out["air"] = s.state()
        if case["pore"]:
            out["pore"] = s.state(1)
    return out


def work(case):
    """State read and written once per step (fields and layer auxiliaries), mean flow read."""
    if case["kind"] == "train":
        it = case["epochs"] * (case["rows"] // case["batch"])
        par = 16 * 64 + 2 * 64 * 64 + 64 * 16 + 208
        return {"bytes": it * (par * 4.0 * 6 + case["batch"] * 48.0), "flops": it * 6.0 * case["batch"] * par}
    nx, ny, nz, w = case["nx"], case["ny"], case["nz"], case["bits"] / 8
    n = nx * ny * nz
    if case["kind"] == "ensemble":
        n = int(n * case["members"] * 0.75 * 0.75 * 0.875)
        nx, ny = 0.75 * nx, 0.75 * ny
    slabs = n * (case["pml"] + 1) * (0 if case.get("walls") else 2 / nx + (1 if case["tdbc"] else 2) / ny)
    slabs += n * (case["pml"] + 1) / nz
    pore = n / nz * case["pore"] * (0.6 if case["kind"] == "ensemble" else 1)
    words = 8 * (n + pore + slabs) + (n if case["wind"] else 0)
    flop = (27 + (14 if case["hills"] else 0) + (40 if case["wind"] else 0)) * n + 30 * pore + 25 * slabs
    if case["scheme"] == "rk4":
        flop = 4 * (flop + 16 * n)
    return {"bytes": float(case["steps"] * words * w), "flops": float(case["steps"] * flop)}


# ------------------------------------------------------------------ the same step in 64-bit torch
class _Domain:
    """One domain's FB_p_v or RK4 step on dense 64-bit tensors, fields [k, j, i]."""

    def __init__(self, p, device):
        self.p, self.dev = p, device
        self.shape = (p["nz"], p["ny"], p["nx"])
        self.ax = [p["d"] * np.arange(p["nz"]), p["d"] * np.arange(p["ny"]), p["x0"] + p["d"] * np.arange(p["nx"])]
        self.inv, self.dt = 1.0 / p["d"], p["dt"]
        self.Aav = p["c"] ** 2 / GAMMA / p["Pav"]
        self.gP = GAMMA * p["Pav"]
        w, bc = p["pml"], p["bc"]
        low = (bc[1] == 2, bc[3] == 2, bc[5] == 2)    # z y x
        high = (bc[0] == 2, bc[2] == 2, bc[4] == 2)
        self.slab = []  # in the order of the layer terms: x1 x2 y1 y2 z1 z2
        for a in (2, 1, 0):
            n, c = self.shape[a], self.ax[a]
            for hi in (0, 1):
                if not (high if hi else low)[a]:
                    continue
                if hi:
                    t = (c - c[n - w]) / abs(c[n - 1] - c[n - w])
                    act, lo = (n - w, n), n - w - 1
                else:
                    t = (c[w - 1] - c) / abs(c[w - 1] - c[0])
                    act, lo = (0, w), 0
                ta = np.where((np.arange(n) >= act[0]) & (np.arange(n) < act[1]), np.abs(t), 0.0) ** ALPHA
                self.slab.append(dict(a=a, act=act, lo=lo, n=w + 1, s=RESIST * ta, b=1.0 / (1.0 + 25.0 * ta)))
        self.x = [self._t(f) for f in _waves(p)]
        self.q = [[torch.zeros([s["n"] if a == s["a"] else m for a, m in enumerate(self.shape)], dtype=torch.float64,
                               device=device) for _ in range(4)] for s in self.slab]
        self.pore = None
        if p["pore"]:
            kp = p["pore"] + 2
            self.pz = p["d"] * (np.arange(kp) - (kp - 2.0))
            gc = 4.0 * math.log(2.0) / p["width"] ** 2
            zs = p["src"][2] + self._hill(p["src"][0], p["src"][1])
            h = self._hill(self.ax[2][None, :], self.ax[1][:, None])
            r2 = (((self.ax[2] - p["src"][0]) ** 2)[None, None, :] + ((self.ax[1] - p["src"][1]) ** 2)[None, :, None] +
                  (self.pz[:, None, None] + h[None] - zs) ** 2)
            self.pore = [torch.zeros(r2.shape, dtype=torch.float64, device=device) for _ in range(3)] + [self._t(np.exp(-gc * r2))]
            rho_e = p["tort"] / p["porosity"] / self.Aav
            self.p_eff, self.p_beta, self.p_gama = 1 / rho_e, p["sigma"] * p["dt"] / rho_e, p["dt"] * self.gP / p["porosity"]
        rho = GAMMA * p["Pav"] / 340.29 ** 2
        self.td_z = rho * 340.29 * math.sqrt(p["tort"]) / p["porosity"]
        self.td_tb = p["dt"] / (GAMMA * rho * p["tort"] / p["sigma"] / p["porosity"])
        self.psi = torch.zeros(6, p["nz"], p["nx"], dtype=torch.float64, device=device)
        self.gpsi = torch.zeros(max(1, p["poles"]), p["ny"], p["nx"], dtype=torch.float64, device=device)
        self.frame(0)

    def _t(self, a):
        return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=self.dev)

    def _hill(self, x, y):
        h = 0.0 * x + 0.0 * y
        for x0, y0, a, s in self.p["hill"]:
            h = h + a * np.exp(-((x - x0) ** 2 + (y - y0) ** 2) / (2.0 * s * s))
        return h

    def frame(self, n):
        """Coordinates, metric and wind of moving frame n; its shift of state and layers."""
        p, sh = self.p, self.p.get("shift", 0)
        if n:
            for f in self.x + (self.pore or []):
                self._shift(f, 1)
            self.x[3][:, 0] = self.x[3][:, 1]
            if self.pore:
                self.pore[3][:, 0] = self.pore[3][:, 1]
            for s, q in zip(self.slab, self.q):
                for f in q:
                    self._shift(f, 1, s["lo"] if s["a"] == 1 else 0, s["a"] == 1)
        else:
            for q in self.q:
                for f in q:
                    f.zero_()
        x, y = self.ax[2][None, :], (self.ax[1] + n * sh * p["d"])[:, None]
        h = self._hill(x, y)
        D = self.ax[0][-1]
        hx, hy = np.zeros_like(h), np.zeros_like(h)
        hx[:, 1:-1] = (h[:, 2:] - h[:, :-2]) * self.inv * 0.5
        hy[1:-1] = (h[2:] - h[:-2]) * self.inv * 0.5
        one = [(np.concatenate([[0], (c[2:] - c[:-2]) * self.inv * 0.5, [0]])) for c in self.ax]
        I = (slice(1, -1),) * 3
        tk = (D - self.ax[0]) / D
        zz = one[0][:, None, None] * (1.0 - h / D)[None]
        with np.errstate(divide="ignore", invalid="ignore"):
            self.mx = self._t((1.0 / one[2])[None, None, 1:-1])
            self.my = self._t((1.0 / one[1])[None, 1:-1, None])
            self.mz = self._t((1.0 / zz)[I])
            self.zx = self._t((-(hx[None] * tk[:, None, None]) / (one[2][None, None, :] * zz))[I])
            self.zy = self._t((-(hy[None] * tk[:, None, None]) / (one[1][None, :, None] * zz))[I])
            # a layer shifted rigidly with the ground: the porous grid and the ground plane
            z1 = 1.0 / one[0][1]
            self.pzx = self._t((-(hx * z1) / one[2][None, :])[1:-1, 1:-1])
            self.pzy = self._t((-(hy * z1) / one[1][:, None])[1:-1, 1:-1])
            self.pmz = z1
        self.V = None
        if p["wind"]:
            zg = self.ax[0][:, None, None] + h[None] * (tk - tk[0])[:, None, None]
            with np.errstate(divide="ignore", invalid="ignore"):
                self.V = self._t(np.where(zg > 0.02, p["ustar"] / 0.41 * np.log(zg / 0.02), 0.0))

    def _shift(self, f, ax, lo=0, layer=False):
        """The frame's shift along y of one field (or of a y layer that starts at plane lo)."""
        p, sh, n = self.p, self.p["shift"], f.shape[1]
        old = f.clone()
        tj = p["ny"] - (sh + 1)
        for jj in range(n):
            j = lo + jj
            if j < tj + 1 and j + sh < p["ny"] - 1:
                f[:, jj] = old[:, jj + sh] if jj + sh < n else 0.0
            elif j >= tj + 1:
                f[:, jj] = 0.0

    # ---- differences on the interior; sl: a region of it (slices of the whole grid)
    @staticmethod
    def _at(f, sl, off, lo=None):
        idx = []
        for a, s in enumerate(sl):
            b = 0 if lo is None or lo[0] != a else lo[1]
            idx.append(slice(s.start + off[a] - b, s.stop + off[a] - b))
        return f[tuple(idx)]

    def _m(self, m, sl):
        return m[tuple(slice(None) if m.shape[a] == 1 else slice(s.start - 1, s.stop - 1) for a, s in enumerate(sl))]

    def _d(self, f, ax, sl, back=False, lo=None):
        """d/dX, d/dY or d/dZ of f, forward (or backward) with the grid's metric."""
        def diff(a):
            o = [0, 0, 0]
            o[a] = -1 if back else 1
            v = self._at(f, sl, o, lo) - self._at(f, sl, (0, 0, 0), lo)
            return (-v if back else v) * self.inv
        if ax == 0:
            return self._m(self.mz, sl) * diff(0)
        v = self._m(self.my if ax == 1 else self.mx, sl) * diff(ax)
        if self.p["hills"]:
            v = v + self._m(self.zy if ax == 1 else self.zx, sl) * diff(0)
        return v

    def _regions(self):
        """Interior parts of the active layer planes, and the pairs of layers that overlap."""
        inner = [(1, n - 1) for n in self.shape]
        regs = []
        for s in self.slab:
            r = list(inner)
            r[s["a"]] = (max(1, s["act"][0]), min(self.shape[s["a"]] - 1, s["act"][1]))
            regs.append([slice(*x) for x in r])
        pairs = []
        for m, s in enumerate(self.slab):
            for n, t in enumerate(self.slab):
                if (t["a"], n) > (s["a"], m) and t["a"] != s["a"]:
                    sl = [slice(max(x.start, y.start), min(x.stop, y.stop)) for x, y in zip(regs[m], regs[n])]
                    if all(x.stop > x.start for x in sl):
                        pairs.append((m, n, sl))  # m: the y or z layer, n: the x (or y) layer
        return regs, pairs

    def _prof(self, s, sl, which):
        a = s["a"]
        v = s["s"] if which == "s" else (1 - s["b"] if which == "c" else s["b"] - 1)
        shape = [1, 1, 1]
        shape[a] = -1
        return self._t(v[sl[a]].reshape(shape))

    def dp(self, x, q, central):
        """dt times the pressure's rate of change on the interior."""
        u, v, w, p = x
        I = [slice(1, n - 1) for n in self.shape]
        dt = self.dt
        ddx, ddy, ddz = self._d(u, 2, I), self._d(v, 1, I), self._d(w, 0, I)
        r = -self.gP * dt * (ddx + ddy + ddz)
        if self.V is not None:
            r = r - dt * self._at(self.V, I, (0, 0, 0)) * self._c(p, 1, I)
            r = r - GAMMA * dt * self._at(p, I, (0, 0, 0)) * self._c(self.V, 1, I)
        whole = {2: ddx, 1: ddy, 0: ddz}
        regs, pairs = self._regions()
        for s, qs, sl in zip(self.slab, q, regs):
            lo = (s["a"], s["lo"])
            inner = tuple(slice(x.start - 1, x.stop - 1) for x in sl)
            rest = sum(self._d(qs[2 - a], a, sl, lo=lo) for a in (2, 1, 0) if a != s["a"])
            r[inner] += dt * (self._prof(s, sl, "c") * self.gP * whole[s["a"]][inner] -
                              self._prof(s, sl, "s") * (self._at(p, sl, (0, 0, 0)) + self.gP * rest))
        for m, n, sl in pairs:
            s, t, qt = self.slab[m], self.slab[n], q[n]
            lo = (t["a"], t["lo"])
            so, st = self._prof(s, sl, "s"), self._prof(t, sl, "s")
            own = self._prof(t, sl, "d") * so * self._d(qt[2 - t["a"]], t["a"], sl, lo=lo)
            other = self._prof(s, sl, "d") * st * self._d(qt[2 - s["a"]], s["a"], sl, lo=lo)
            r[tuple(slice(x.start - 1, x.stop - 1) for x in sl)] -= dt * (self._at(qt[3], sl, (0, 0, 0), lo) * st * so + self.gP * (own + other))
        return r

    def _c(self, f, ax, sl):
        """Central difference of a field with the metric."""
        return 0.5 * (self._d(f, ax, sl) + self._d(f, ax, sl, back=True))

    def duvw(self, x, p, q, qp):
        """dt times the velocities' rates of change; p and qp the pressure and its auxiliaries."""
        I = [slice(1, n - 1) for n in self.shape]
        dt, A = self.dt, self.Aav
        grad = {a: self._d(p, a, I, back=True) for a in (2, 1, 0)}
        out = [-A * dt * grad[2 - f] for f in range(3)]
        if self.V is not None:
            Vc = self._at(self.V, I, (0, 0, 0))
            for f in range(3):
                out[f] = out[f] - dt * Vc * self._c(x[f], 1, I)
                out[1] = out[1] - dt * self._at(x[f], I, (0, 0, 0)) * self._c(self.V, 2 - f, I)
        regs, pairs = self._regions()
        for s, qs, sl in zip(self.slab, qp, regs):
            lo = (s["a"], s["lo"])
            inner = tuple(slice(y.start - 1, y.stop - 1) for y in sl)
            sg, cg = self._prof(s, sl, "s"), self._prof(s, sl, "c")
            for f in range(3):
                own = self._at(x[f], sl, (0, 0, 0))
                if 2 - f == s["a"]:
                    out[f][inner] += dt * (cg * A * grad[2 - f][inner] - sg * own)
                else:
                    out[f][inner] -= dt * sg * (own + A * self._d(qs, 2 - f, sl, back=True, lo=lo))
        for m, n, sl in pairs:
            s, t = self.slab[m], self.slab[n]
            lo = (t["a"], t["lo"])
            inner = tuple(slice(y.start - 1, y.stop - 1) for y in sl)
            so, st = self._prof(s, sl, "s"), self._prof(t, sl, "s")
            for f in range(3):
                v = self._at(q[n][f], sl, (0, 0, 0), lo) * st * so
                if 2 - f == t["a"]:
                    v = v + self._prof(t, sl, "d") * so * A * self._d(qp[n], 2 - f, sl, back=True, lo=lo)
                elif 2 - f == s["a"]:
                    v = v + self._prof(s, sl, "d") * st * A * self._d(qp[n], 2 - f, sl, back=True, lo=lo)
                out[f][inner] -= dt * v
        return out

    def pore_div(self, y):
        c = (slice(1, -1),) * 3
        dz = [(f[2:, 1:-1, 1:-1] - f[c]) * self.inv for f in y[:3]]
        r = self.mx * (y[0][1:-1, 1:-1, 2:] - y[0][c]) * self.inv + self.my * (y[1][1:-1, 2:, 1:-1] - y[1][c]) * self.inv + self.pmz * dz[2]
        return r + self.pzx * dz[0] + self.pzy * dz[1]

    def pore_grad(self, p):
        c = (slice(1, -1),) * 3
        dz = (p[c] - p[:-2, 1:-1, 1:-1]) * self.inv
        return [self.mx * (p[c] - p[1:-1, 1:-1, :-2]) * self.inv + self.pzx * dz,
                self.my * (p[c] - p[1:-1, :-2, 1:-1]) * self.inv + self.pzy * dz, self.pmz * dz]

    # ---- faces, in the reference's order: N E W F B, then the ground
    def faces_p(self, p, pp):
        def sides(f, top):
            if top:
                f[-1] = f[-2]
            else:
                f[0] = f[1]
            f[:, -1] = 15 / 8 * f[:, -2] - 5 / 4 * f[:, -3] + 3 / 8 * f[:, -4]
            f[:, 0] = f[:, 1]
            f[:, :, 0] = f[:, :, 1]
            f[:, :, -1] = f[:, :, -2]
        sides(p, True)
        if pp is not None:
            sides(pp, False)
            p[0] = pp[-2]
            pp[-1] = p[1]
        elif not self.p["poles"]:
            p[0] = p[1]

    def faces_v(self, x, y, vt=None):
        def sides(u, v, w, top):
            e, s = (-1, -2) if top else (0, 1)
            u[e], v[e], w[e] = u[s], v[s], 0.0
            u[:, -1], w[:, -1] = u[:, -2], w[:, -2]
            v[:, -1] = 0.0 if vt is None else vt
            u[:, 0], v[:, 0], w[:, 0] = u[:, 1], 0.0, w[:, 1]
            u[:, :, 0], v[:, :, 0], w[:, :, 0] = 0.0, v[:, :, 1], w[:, :, 1]
            u[:, :, -1], v[:, :, -1], w[:, :, -1] = 0.0, v[:, :, -2], w[:, :, -2]
        sides(*x[:3], True)
        if y is not None:
            sides(*y[:3], False)
            for a, b in zip(x[:3], y[:3]):
                a[0] = b[-2]
                b[-1] = a[1]
        elif not self.p["poles"]:
            x[0][0], x[1][0], x[2][0] = x[0][1], x[1][1], 0.0

    def _aux(self, f, k):
        """Field k restricted to each layer's planes."""
        out = []
        for s in self.slab:
            out.append(f[tuple(slice(s["lo"], s["lo"] + s["n"]) if a == s["a"] else slice(None) for a in range(3))])
        return out

    def fb_step(self):
        p, x, q, dt, c = self.p, self.x, self.q, self.dt, (slice(1, -1),) * 3
        new = [f.clone() for f in x]
        new[3][c] += self.dp(x, q, False)
        pn = None
        if self.pore:
            pn = [f.clone() for f in self.pore]
            pn[3][c] -= self.p_gama * self.pore_div(self.pore)
        g = (0, slice(1, -1), slice(1, -1))
        if p["poles"]:
            rho_e = p["tort"] / p["porosity"] / self.Aav
            eff, gama, ib = 1 / rho_e, dt * self.gP / p["porosity"], 1 / (p["sigma"] * dt / rho_e + 1)
            dz = [(f[1, 1:-1, 1:-1] - f[g]) * self.inv for f in x]
            div = (self.mx[0] * (x[0][0, 1:-1, 2:] - x[0][g]) * self.inv + self.pzx * dz[0] +
                   self.my[0] * (x[1][0, 2:, 1:-1] - x[1][g]) * self.inv + self.pzy * dz[1] + self.pmz * dz[2])
            new[3][g] = x[3][g] - gama * div
        self.faces_p(new[3], pn[3] if pn else None)
        qp = [a[3] + dt * f for a, f in zip(q, self._aux(new[3], 3))]
        for f, v in zip(range(3), self.duvw(x, new[3], q, qp)):
            new[f][c] += v
        if self.pore:
            ib = 1 / (1 + self.p_beta)
            for f, gr in zip(range(3), self.pore_grad(pn[3])):
                pn[f][c] = ib * (self.pore[f][c] - dt * self.p_eff * gr)
        if p["poles"]:
            P = new[3]
            pz = (P[1, 1:-1, 1:-1] - P[g]) * self.inv
            gx = self.mx[0] * (P[g] - P[0, 1:-1, :-2]) * self.inv + self.pzx * pz
            gy = self.my[0] * (P[g] - P[0, :-2, 1:-1]) * self.inv + self.pzy * pz
            new[0][g] = ib * (x[0][g] - dt * eff * gx)
            new[1][g] = ib * (x[1][g] - dt * eff * gy)
            tb = dt / p["tau"]
            a, r = (self._t([v[n] for v in p["pole"]])[:, None, None] for n in (0, 1))
            dec = torch.exp(-r * tb)
            cpl = 2 * dt * eff * self.pmz * self.inv
            P8 = self.gpsi[:, 1:-1, 1:-1]
            wn = (x[2][g] - cpl * (P[g] - p["zinf"] * (dec * P8).sum(0))) * ib / (1 + ib * cpl * p["zinf"] * (1 + tb * float(a.sum())))
            new[2][g] = wn
            self.gpsi[:, 1:-1, 1:-1] = dec * P8 - a * wn * tb
        vt = None
        if p["tdbc"]:
            tb = self.td_tb
            dec = self._t([math.exp(-r * tb) for r in TD_R])[:, None, None]
            vt = (new[3][:, -1] / self.td_z - (dec * self.psi).sum(0)) / (1 + sum(TD_A) * tb)
            self.psi = dec * self.psi + self._t(TD_A)[:, None, None] * vt * tb
        self.faces_v(new, pn, vt)
        self.q = [[a[f] + dt * aux for f, aux in zip(range(3), [self._aux(new[f], f)[m] for f in range(3)])] + [qp[m]]
                  for m, a in enumerate(q)]
        self.x, self.pore = new, pn

    def rk_step(self):
        dt, c = self.dt, (slice(1, -1),) * 3
        x0, y0, q0 = self.x, self.pore, self.q
        xs, ys, qs = x0, y0, q0
        acc, qacc = [f.clone() for f in x0], [[f.clone() for f in q] for q in q0]
        if y0:
            E, E2 = math.exp(-self.p_beta), math.exp(-0.5 * self.p_beta)
            yacc = [E * f for f in y0[:3]] + [y0[3].clone()]
        for st in range(4):
            a, b = (0.5, 0.5, 1.0, 0.0)[st], (1 / 6, 1 / 3, 1 / 3, 1 / 6)[st]
            k = self.duvw(xs, xs[3], qs, [q[3] for q in qs]) + [self.dp(xs, qs, True)]
            nx = [f.clone() for f in (x0 if st < 3 else acc)]
            for f in range(4):
                nx[f][c] += (a if st < 3 else b) * k[f]
                acc[f][c] += b * k[f]
            ny = None
            if y0:
                N = [-dt * self.p_eff * gr for gr in self.pore_grad(ys[3])]
                kp = -self.p_gama * self.pore_div(ys)
                ny = [f.clone() for f in y0]
                for f in range(3):
                    yacc[f][c] += (E / 6, E2 / 3, E2 / 3, 1 / 6)[st] * N[f]
                    if st < 3:
                        ny[f][c] = (E2, E2, E)[st] * y0[f][c] + (0.5 * E2, 0.5, E2)[st] * N[f]
                    else:
                        ny[f][c] = yacc[f][c]
                yacc[3][c] += b * kp
                ny[3][c] = y0[3][c] + a * kp if st < 3 else yacc[3][c]
            self.faces_p(nx[3], ny[3] if ny else None)
            self.faces_v(nx, ny)
            nq = []
            for m in range(len(self.slab)):
                row = []
                for f in range(4):
                    rate = dt * self._aux(xs[f], f)[m]
                    qacc[m][f] += b * rate
                    row.append(q0[m][f] + a * rate if st < 3 else qacc[m][f])
                nq.append(row)
            xs, ys, qs = nx, ny, nq
        self.x, self.pore, self.q = xs, ys, qs

    def steps(self, n, shift=0):
        """n steps; the receivers sample the pressure before each (0 outside the frame)."""
        i, j, k = (torch.as_tensor(v.copy(), device=self.dev) for v in self.p["rec"].T)
        j = j - shift
        ok = (j > 0) & (j < self.p["ny"] - 1)
        out = []
        for _ in range(n):
            out.append(torch.where(ok, self.x[3][k, j.clamp(0, self.p["ny"] - 1), i], 0.0))
            if self.p["scheme"] == "rk4":
                self.rk_step()
            else:
                self.fb_step()
        return torch.stack(out)


def _train_exact(case, seed):
    x, t, w = (a.astype(np.float64) for a in _training(case, seed))
    dims = ((64, 16), (64, 64), (64, 64), (16, 64))
    rows, batch = case["rows"], min(case["batch"], case["rows"])
    x = np.pad(x, ((0, 0), (0, 12)))
    w, m, v = w.copy(), np.zeros_like(w), np.zeros_like(w)
    order, st, step, mse = list(range(rows)), (7 + 0x9E3779B97F4A7C15) % 2 ** 64, 0, 0.0
    c = math.sqrt(2 / math.pi)
    for _ in range(case["epochs"]):
        for i in range(rows - 1, 0, -1):
            st = (st * 6364136223846793005 + 1442695040888963407) % 2 ** 64
            j = (st >> 33) % (i + 1)
            order[i], order[j] = order[j], order[i]
        for b0 in range(0, rows - batch + 1, batch):
            pick = order[b0:b0 + batch]
            a, off, keep = x[pick], 0, []
            for n, (o, i) in enumerate(dims):
                W, b = w[off:off + o * i].reshape(o, i), w[off + o * i:off + o * i + o]
                z = a @ W.T + b
                keep.append((off, W, a, z))
                off += o * i + o
                a = 0.5 * z * (1 + np.tanh(c * (z + 0.044715 * z ** 3))) if n < 3 else z
            e = a[:, :8] - t[pick]
            mse = float((e ** 2).mean())
            dz, g = np.pad(2 * e / e.size, ((0, 0), (0, 8))), np.zeros_like(w)
            for n in (3, 2, 1, 0):
                off, W, a, z = keep[n]
                if n < 3:
                    th = np.tanh(c * (z + 0.044715 * z ** 3))
                    dz = dz * (0.5 * (1 + th) + 0.5 * z * (1 - th * th) * c * (1 + 3 * 0.044715 * z * z))
                g[off:off + W.size], g[off + W.size:off + W.size + W.shape[0]] = (dz.T @ a).ravel(), dz.sum(0)
                dz = dz @ W
            step += 1
            m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
            w = w - 2e-3 * (m / (1 - 0.9 ** step)) / (np.sqrt(v / (1 - 0.999 ** step)) + 1e-8)
    return {"params": w, "mse": mse}


def exact(case, seed):
    if case["kind"] == "train":
        return _train_exact(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    with torch.no_grad():
        if case["kind"] == "ensemble":
            parts = [_Domain(_inputs(case, seed, m), dev).steps(case["steps"]) for m in range(case["members"])]
            return {"series": torch.cat(parts, dim=1)}
        p = _inputs(case, seed)
        d = _Domain(p, dev)
        if case["kind"] == "frames":
            parts, done, mf, last = [], 0, 0, 4
            while done < p["steps"]:
                per = p["shift"] * p["d"] / p["c"] / p["dt"]
                n = int((p["ny"] - 1) * p["d"] / p["c"] / p["dt"] * 0.4) if mf == 0 else int(per)
                n = p["steps"] - done if mf == last else min(n, p["steps"] - done)
                d.frame(mf)
                parts.append(d.steps(n, mf * p["shift"]))
                done, mf = done + n, mf + 1
            return {"series": torch.cat(parts)}
        out = {"series": d.steps(p["steps"])}
        if p["state"]:
            out["air"] = d.x
            if p["pore"]:
                out["pore"] = d.pore
        return out
