"""Performance cases of the PIC step: what a user of the package has the GPU
do, through the public classes, over the range of sizes, modes, precisions
and plasma layouts that the workloads of chimeracl_amd.config span.

Kinds of case (field "kind"):
  step       whole PIC steps of a laser-plasma run: PIC_loop.step(), or
             PIC_loop.run(n) replaying captured steps
  deposit    the particle half of a step on its own: half push, sort, J,
             half push, sort, rho (electrons and immobile ions)
  gather     field gather + Boris push of the sorted electrons
  transform  rho and J to spectral space with smoothing, E and B back
  update     density gradient, PSATD advance + edge damping, B = rot(G)/w^2
  gradient   a differentiable run: forward steps and the reverse sweep
  setup      a new Solver (all of its tables) and the laser pulse

Other fields: precision ("f64" or "mixed") and, for mixed, the DHT product
("bf16x3" or "f32"); grid nx, nr and highest mode m; npc particles per
loading cell; drift, the distance in cells that the electrons have moved
since their memory order last followed the cells (0: just realigned).

exact(case, seed) computes the same outputs in float64 with plain torch and
numpy: Bessel functions from their integral, roots by Newton's method, the
DHT as a matrix inverse, FFTs and products from torch, deposits by index_add.
"""
import math

import numpy as np
import torch

DZ, DR, DENS = 0.02, 0.1, 0.002
COMPS = ("x", "y", "z")


def _case(name, kind, precision, nx, nr, m, npc=0, drift=0.0, dht="bf16x3", steps=0, graph=False,
          align=0):
    c = {"kind": kind, "precision": precision, "nx": nx, "nr": nr, "m": m, "npc": npc,
         "drift": drift, "dht": dht, "steps": steps, "graph": graph, "align": align}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a first try of a run: small box, default loop options, one step at
        # a time; launches and host work count
        _case("step_small_f64", "step", "f64", 256, 64, 1, 16, steps=1),
        # the production run in its plain form: 4096 x 512, modes 0..2,
        # captured steps, electrons realigned every 20 steps
        _case("step_large_f64", "step", "f64", 4096, 512, 2, 32, steps=4, graph=True, align=20),
        # the medium run in its mixed form
        _case("step_mid_mixed", "step", "mixed", 2048, 256, 1, 32, steps=4, graph=True, align=20),
        # particle half of the production step, some steps after a realignment
        _case("deposit_large_mixed", "deposit", "mixed", 4096, 512, 2, 32, drift=0.5),
        # the same at odd sizes: 1024 x 201 grid, 15 particles per cell, memory
        # order far behind the cells (no realignment)
        _case("deposit_odd_f64", "deposit", "f64", 1024, 201, 1, 15, drift=3.0),
        # gather + push, production size
        _case("gather_large_mixed", "gather", "mixed", 4096, 512, 2, 32, drift=0.5),
        # gather + push of a small run
        _case("gather_small_f64", "gather", "f64", 512, 128, 1, 16, drift=0.5),
        # Fourier-Bessel transforms both ways
        _case("transform_large_mixed", "transform", "mixed", 4096, 512, 2),
        _case("transform_mid_f64", "transform", "f64", 2048, 256, 1),
        # spectral field update
        _case("update_mid_mixed", "update", "mixed", 1024, 256, 1),
        # gradients of a small differentiable run
        _case("gradient_f64", "gradient", "f64", 1024, 128, 1, 16, steps=4),
        # a new simulation: tables and laser, mixed form
        _case("setup_mixed", "setup", "mixed", 1024, 256, 1),
    ]


def draw(rng):
    kind = rng.choice(["step", "deposit", "gather", "transform", "update", "gradient", "setup"])
    prec = rng.choice(["f64", "mixed"])
    dht = rng.choice(["bf16x3", "bf16x3", "f32"]) if prec == "mixed" else "bf16x3"
    grad = kind == "gradient"
    m = rng.choice([0, 1, 1, 1, 2, 2, 3]) if not grad else rng.choice([1, 1, 2])
    nx = 2 ** rng.randint(6, 11 if grad else 12)
    nr = int(round(math.exp(rng.uniform(math.log(24), math.log(256 if grad else 512)))))
    while nx * nr * (m + 1) > 4096 * 512 * 3:
        nx //= 2
    npc = int(round(math.exp(rng.uniform(math.log(2), math.log(48)))))
    npc = max(1, min(npc, int((4e6 if grad else 6e7) / (nx * nr))))
    drift = rng.choice([0.0, 0.5, 0.5, 3.0])
    if kind in ("transform", "update", "setup"):
        return _case(None, kind, prec, nx, nr, m, dht=dht)
    if kind in ("deposit", "gather"):
        return _case(None, kind, prec, nx, nr, m, npc, drift, dht)
    if grad:
        return _case(None, kind, prec, nx, nr, m, npc, 0.0, dht, steps=rng.choice([2, 3, 4]))
    graph = rng.choice([False, True, True])
    return _case(None, kind, prec, nx, nr, m, npc, drift, dht, steps=rng.choice([2, 3]) if graph else 1,
                 graph=graph, align=rng.choice([0, 20]) if graph else 0)


# ---------------------------------------------------------------- inputs
def _grid_cfg(c):
    nx, nr = c["nx"], c["nr"]
    return {"Xmin": -(nx - 1) * DZ, "Xmax": 0.0, "Nx": nx, "Rmin": 0.0, "Rmax": DR * (nr - 1.5),
            "Nr": nr, "M": c["m"], "dt": DZ, "DampCells": min(50, nx // 16)}


def _laser_cfg(c, seed):
    """A pulse that fits the box; its amplitude varies with the seed."""
    lx, lr = c["nx"] * DZ, c["nr"] * DR
    x0 = -min(3.0, 0.3 * lx)
    return {"k0": 1.0, "a0": 2.0 + 0.01 * (seed % 97), "x0": x0, "Lx": min(5.1, 0.25 * lx),
            "R": min(4.0, 0.3 * lr), "x_foc": x0}


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _real(c):
    return torch.float64 if c["precision"] == "f64" else torch.float32


def _off(v, edge, margin):
    """v moved off the band edge +- margin."""
    return torch.where((v - edge).abs() < margin, torch.full_like(v, edge + 2 * margin), v)


def _plasma(c, seed, dp=0.005):
    """Electrons of a run in flight, float64 (already rounded to the run's
    precision): uniformly jittered plasma on the loading cells of
    chimeracl_amd.config.load_plasma, in cell order, then moved by drift
    cells (normally distributed), with thermal momenta dp.  The last half
    loading row and what drifted out of the box are outside the valid
    cells; none lies within a thousandth of a cell of their border."""
    nx, nr, npc = c["nx"], c["nr"], c["npc"]
    g = _gen(seed)
    f8 = dict(dtype=torch.float64, device="cuda")
    ncx, ncr = nx - 3, nr - 2
    n = ncx * ncr * npc
    xmin = -(nx - 1) * DZ
    cell = torch.arange(ncx * ncr, device="cuda").repeat_interleave(npc)
    fx = 1 + cell % ncx + torch.rand(n, generator=g, **f8)        # in cells from Xmin
    fr = cell // ncx + torch.rand(n, generator=g, **f8)           # r / dr
    key = torch.floor(fr + 0.5).long() * nx + torch.floor(fx).long()
    order = torch.argsort(key, stable=True)
    fx, fr = fx[order], fr[order]
    del cell, key, order
    if c["drift"]:
        fx += c["drift"] * torch.randn(n, generator=g, **f8)
        fr = (fr + c["drift"] * torch.randn(n, generator=g, **f8)).abs()
    fx = _off(_off(fx, 1.0, 1e-3), nx - 2.0, 1e-3)
    fr = _off(fr, nr - 2.5, 1e-3)
    th = 2 * math.pi * torch.rand(n, generator=g, **f8)
    rnd = lambda t: t.to(_real(c)).double()
    r = fr * DR
    out = {"x": rnd(xmin + DZ * fx), "y": rnd(r * torch.sin(th)), "z": rnd(r * torch.cos(th)),
           "w": rnd(2 * math.pi * DZ * DR * DENS / npc * r)}
    del fx, fr, th, r
    for k in ("px", "py", "pz"):
        out[k] = rnd(dp * torch.randn(n, generator=g, **f8))
    out["g_inv"] = rnd(1 / torch.sqrt(1 + out["px"] ** 2 + out["py"] ** 2 + out["pz"] ** 2))
    return out


def _planes(c, names, seed, spectral, amp=None):
    """Random real-space or spectral planes {name_m<m>: float64 / complex128},
    rounded to the run's precision; higher modes weaker, as in a run."""
    g = _gen(seed)
    nx, nr = c["nx"], c["nr"]
    shp = (nr - 1, nx) if spectral else (nr, nx)
    out = {}
    for n in names:
        for m in range(c["m"] + 1):
            s = 0.3 ** m * ((amp or {}).get(n[0], 1.0))
            re = (s * torch.randn(shp, generator=g, dtype=torch.float64, device="cuda")).to(_real(c)).double()
            if m == 0 and not spectral:
                out[f"{n}_m{m}"] = re
                continue
            im = (s * torch.randn(shp, generator=g, dtype=torch.float64, device="cuda")).to(_real(c)).double()
            out[f"{n}{'_fb' if spectral else ''}_m{m}"] = torch.complex(re, im)
    return out


_AMP = {"E": 1.0, "B": 1.0, "G": 60.0, "J": 0.01, "r": 0.01, "d": 0.05}


def _vec(*flds):
    return [f + k for f in flds for k in COMPS]


# ---------------------------------------------------------------- the framework's side
def _comm(c):
    from chimeracl_amd import Communicator
    return Communicator(precision=c["precision"], dht=c["dht"])


def _species_cfg(c, charge):
    cfg = {"Nppc": (c["npc"], 1, 1), "dx": DZ, "dr": DR, "dt": DZ, "dens": DENS, "charge": charge}
    return dict(cfg, Immobile=True) if charge > 0 else cfg


class _Source:
    def __init__(self, arrays):
        self.DataDev = {k + "_new": v for k, v in arrays.items()}


def _species(c, comm, plasma):
    import chimeracl_amd as CA
    eons, ions = CA.Particles(_species_cfg(c, -1), comm), CA.Particles(_species_cfg(c, 1), comm)
    eons.add_particles(source=_Source(plasma))
    ions.add_particles(source=_Source(plasma))
    return eons, ions


def _put(solver, planes):
    for k, v in planes.items():
        solver.DataDev[k].copy_(v)


def prepare(case, seed):
    import chimeracl_amd as CA
    c = case
    kind = c["kind"]
    if kind == "setup":
        return {"case": c, "cfg": _grid_cfg(c), "laser": _laser_cfg(c, seed), "comm": _comm(c)}
    if kind == "gradient":
        from chimeracl_amd.adjoint import DiffPIC
        kn = _knots(c, seed)
        sim = DiffPIC(_grid_cfg(c), _laser_cfg(c, seed), (_species_cfg(c, -1), _species_cfg(c, 1)),
                      _plasma(c, seed, dp=0.0), kn[0], _comm(c), ckpt=2)
        return {"case": c, "sim": sim, "knots": kn[1], "laser": _laser_cfg(c, seed),
                "rgrid": sim.solver.Args["Rgrid"]}
    comm = _comm(c)
    solver = CA.Solver(_grid_cfg(c), comm)
    st = {"case": c, "solver": solver}
    if kind in ("step", "deposit", "gather"):
        st["eons"], st["ions"] = _species(c, comm, _plasma(c, seed))
    if kind == "step":
        CA.add_gausian_pulse(solver, _laser_cfg(c, seed))
        st["loop"] = CA.PIC_loop(solvers=[solver], species=[st["eons"], st["ions"]],
                                 graph=c["graph"], align_every=c["align"])
    elif kind == "gather":
        _put(solver, _planes(c, _vec("E", "B"), seed + 1, False))
        st["eons"].sort_parts(solver)
    elif kind == "transform":
        _put(solver, _planes(c, ["rho"] + _vec("J"), seed, False))
        _put(solver, _planes(c, _vec("E", "B"), seed + 1, True))
    elif kind == "update":
        _put(solver, _planes(c, ["rho"] + _vec("E", "G", "J", "dN1"), seed, True, _AMP))
    return st


def _knots(c, seed):
    x = np.linspace(-(c["nx"] - 1) * DZ, 0.0, 32)
    return x, 1.0 + 0.2 * np.random.default_rng(int(seed)).uniform(-1, 1, 32)


def _got(solver, names, spectral=False):
    M = solver.Args["M"]
    return {f"{n}_m{m}": solver.DataDev[f"{n}{'_fb' if spectral else ''}_m{m}"]
            for n in names for m in range(M + 1)}


def _parts(eons, names):
    return {k: eons.DataDev[k] for k in names}


def run(state):
    import chimeracl_amd as CA
    c = state["case"]
    kind = c["kind"]
    if kind == "setup":
        solver = CA.Solver(dict(state["cfg"]), state["comm"])
        CA.add_gausian_pulse(solver, dict(state["laser"]))
        out = _got(solver, _vec("E", "B"))
        out.update({k + str(m): solver.DataDev[k + str(m)] for k in
                    ("DHT_m", "DHT_inv_m", "dDHT_plus_m", "dDHT_minus_m") for m in range(c["m"] + 1)})
        return out
    if kind == "gradient":
        from chimeracl_amd import adjoint as A
        dt = _real(c)
        a0, w0 = (torch.tensor(state["laser"][k], dtype=dt, requires_grad=True) for k in ("a0", "R"))
        kn = torch.tensor(state["knots"], dtype=dt, requires_grad=True)
        out = A.run(state["sim"], a0, w0, kn, c["steps"])
        loss = A.objective_wake_energy(out[3:], state["rgrid"])
        loss = loss + 1e-3 * sum((p.double() ** 2).sum() for p in out[:3])
        loss.backward()
        return {"loss": loss.detach().to(dt), "a0": a0.grad, "w0": w0.grad, "knots": kn.grad}
    solver = state["solver"]
    if kind == "transform":
        solver.fb_transform_smooth(scals=["rho"], vects=["J"])
        solver.fb_transform(vects=["E", "B"], dir=1)
        return [_got(solver, ["rho"] + _vec("J"), True), _got(solver, _vec("E", "B"))]
    if kind == "update":
        solver.field_grad("rho", "dN1", copy_to="dN0")
        solver.damp_edges(("E", "G"), advance_with=("J", "dN0", "dN1"))
        solver.restore_B_fb()
        return _got(solver, _vec("E", "G", "B", "dN0", "dN1"), True)
    eons = state["eons"]
    if kind == "gather":
        solver.gather_and_push([eons])
        return _parts(eons, ("px", "py", "pz", "g_inv"))
    species = [eons, state["ions"]]
    if kind == "deposit":
        for parts in species:
            parts.push_coords(mode="half", grid=solver)
            parts.sort_parts(grid=solver)
        solver.depose_currents(species=species)
        for parts in species:
            parts.push_coords(mode="half", grid=solver)
            parts.sort_parts(grid=solver)
        solver.depose_charge(species=species)
        return [_got(solver, _vec("J") + ["rho"]), _parts(eons, ("x", "y", "z")),
                _parts(eons, ("sort_indx", "cell_offset"))]
    if c["graph"]:
        state["loop"].run(c["steps"])
    else:
        for _ in range(c["steps"]):
            state["loop"].step()
    return [_got(solver, _vec("E", "B", "J") + ["rho"]),
            _parts(eons, ("x", "y", "z", "px", "py", "pz", "g_inv"))]


# ---------------------------------------------------------------- the work of a pass
def work(case):
    c = case
    nx, nr, M, w = c["nx"], c["nr"], c["m"], 8 if c["precision"] == "f64" else 4
    nk = nr - 1
    n = (nx - 3) * (nr - 2) * c["npc"]
    real, spec, tab = nr * nx * w * (1 + 2 * M), 2 * w * nk * nx * (M + 1), w * nk * nx * (M + 1)
    dht = 2 * nk * nk * nx * (1 + 2 * M)           # one field, one direction
    deriv = 2 * nk * nk * 2 * nx * (2 * M + (M > 0) * 1)  # products with dDHT+-: one operand a mode
    fft = 5 * nk * nx * math.log2(nx) * (M + 1)    # one field
    parts = {"push": 200, "deposit": 16 * (2 + 4 * M), "gather": 24 * (2 + 8 * M)}
    update = {"bytes": (1 + 6 + 3 + 3) * spec + 3 * tab + (6 + 6 + 3) * spec,
              "flops": 3 * deriv + 12 * fft + 6 * 2 * 30 * nk * nx * (M + 1)}
    tr = {"bytes": 10 * (real + spec) + tab, "flops": 10 * (dht + fft)}
    step = {"bytes": n * (21 * w + 24) + 20 * real + 53 * spec + 3 * tab,
            "flops": tr["flops"] + update["flops"] + n * (parts["push"] + 4 * parts["deposit"] + parts["gather"])}
    if c["kind"] == "deposit":
        return {"bytes": n * (15 * w + 4) + 4 * (nx - 1) * nk + 4 * real,
                "flops": n * 5 * parts["deposit"]}
    if c["kind"] == "gather":
        return {"bytes": n * (10 * w + 4) + 6 * real, "flops": n * (parts["gather"] + parts["push"])}
    if c["kind"] == "transform":
        return tr
    if c["kind"] == "update":
        return update
    if c["kind"] == "setup":
        return {"bytes": 8 * (5 * nk * nx + 4 * nk * nk) * (M + 1) + 6 * real,
                "flops": (2 + 4) * nk ** 3 * (M + 1) + 7 * (dht + fft) + 2 * deriv}
    k = c["steps"] * (4 if c["kind"] == "gradient" else 1)  # forward, recomputation, reverse
    return {"bytes": k * step["bytes"], "flops": k * step["flops"]}


# ---------------------------------------------------------------- float64 values
def _jn(m, x):
    """J_m(x), 0 <= x < 1900: mean of cos(m t - x sin t) over 2048 points of
    a period (aliased terms J_{2048 -+ m} vanish)."""
    t = torch.arange(2048, dtype=torch.float64, device="cuda") * (2 * math.pi / 2048)
    out = torch.zeros_like(x)
    for i in range(0, 1025, 32):   # t and -t pair up: cos(m t) cos(x sin t) + sin(m t) sin(x sin t)
        tt = t[i:min(i + 32, 1025)]
        wt = torch.where((tt == 0) | (tt == math.pi), 1.0, 2.0)
        a = x.unsqueeze(-1) * torch.sin(tt)
        out += (wt * torch.cos(m * tt - a)).sum(-1)
    return out / 2048


def _roots(m, n):
    """First n positive zeros of J_m: McMahon's expansion, then Newton."""
    b = (torch.arange(1, n + 1, dtype=torch.float64, device="cuda") + 0.5 * m - 0.25) * math.pi
    mu = 4.0 * m * m
    x = b - (mu - 1) / (8 * b) - 4 * (mu - 1) * (7 * mu - 31) / (3 * (8 * b) ** 3)
    for _ in range(8):
        x = x - _jn(m, x) / (0.5 * (_jn(m - 1, x) - _jn(m + 1, x)))
    return x


class _Exact:
    """Float64 restatement of the grid and the spectral operators."""

    def __init__(self, c):
        self.c = c
        nx, nr, M = c["nx"], c["nr"], c["m"]
        self.nx, self.nr, self.M = nx, nr, M
        self.xmin = -(nx - 1) * DZ
        dx, dr = (0.0 - self.xmin) / (nx - 1), DR * (nr - 1.5) / (nr - 1.5)
        self.dx, self.dr, self.rmin = dx, dr, -0.5 * dr
        dev = dict(dtype=torch.float64, device="cuda")
        self.f = {}
        if c["kind"] in ("deposit", "gather"):
            self._volumes()
            return
        self._volumes()
        r = self.rmin + dr * torch.arange(1, nr, **dev)
        R = float(r[-1]) + 0.5 * dr
        kr = [_roots(m, nr - 1) / R for m in range(M + 2)]
        self.kx = torch.from_numpy(2 * np.pi * np.fft.fftfreq(nx, dx)).cuda()
        w = [torch.sqrt(self.kx ** 2 + kr[m][:, None] ** 2) for m in range(M + 1)]
        self.w, self.inv, self.dht, self.dp, self.dm = w, [], [], [], []
        for m in range(M + 1):
            inv = _jn(m, r[:, None] * kr[m])
            fwd = torch.from_numpy(np.linalg.inv(inv.cpu().numpy())).cuda()
            self.inv.append(inv)
            self.dht.append(fwd)
            kp, km = kr[m + 1], kr[abs(m - 1)]
            self.dp.append(fwd @ (0.5 * kp * _jn(m, r[:, None] * kp)))
            self.dm.append(fwd @ (0.5 * km * _jn(m, r[:, None] * km)))
        s = lambda k: 1 - torch.sin(0.5 * math.pi * k / k.max()) ** 2
        self.smooth = [s(self.kx) * s(kr[m])[:, None] for m in range(M + 1)]
        a = self.xmin * self.kx
        self.phase = torch.complex(torch.cos(a), -torch.sin(a))
        nd = min(50, nx // 16)
        z = torch.arange(2 * nd, **dev)
        prof = torch.where(z < nd, 0.0, torch.where(z >= 4 * nd / 3, 1.0, torch.sin(
            0.5 * math.pi * 3.0 * (z - nd + 1) / (nd + 1)) ** 2))
        self.damp = torch.ones(nx, **dev)
        self.damp[:2 * nd] *= prof
        x = torch.arange(nx - 2 * nd + 1, nx, device="cuda")
        self.damp[x] *= prof[nx - x]

    def _volumes(self):
        r = self.rmin + self.dr * torch.arange(self.nr, dtype=torch.float64, device="cuda")
        self.rgrid = r
        self.dv = torch.where(r > 0, 1 / (2 * math.pi * self.dx * self.dr * r), 0.0)

    @staticmethod
    def mul(A, X):
        if not X.is_complex():
            return A @ X.contiguous()
        return torch.complex(A @ X.real.contiguous(), A @ X.imag.contiguous())

    def forward(self, names, smooth=False):
        for n in names:
            for m in range(self.M + 1):
                v = torch.fft.fft(self.mul(self.dht[m], self.f[f"{n}_m{m}"][1:]), dim=1) * self.phase
                self.f[f"{n}_fb_m{m}"] = v * self.smooth[m] if smooth else v

    def backward(self, names):
        for n in names:
            for m in range(self.M + 1):
                v = torch.fft.ifft(self.f[f"{n}_fb_m{m}"] * self.phase.conj(), dim=1)
                v = self.mul(self.inv[m], v.real if m == 0 else v)
                self.f[f"{n}_m{m}"] = torch.cat([torch.zeros_like(v[:1]), v])

    def _below(self, name, m):
        """Mode m - 1 of a spectral field; mode -1 is -conj(F_1(-kx))."""
        if m > 0:
            return self.f[f"{name}_fb_m{m - 1}"]
        v = torch.roll(torch.flip(self.f[f"{name}_fb_m1"], (1,)), 1, 1)
        return -v.conj()

    def grad(self, scl, vec):
        f, M = self.f, self.M
        for m in range(M + 1):
            x = 1j * self.kx * f[f"{scl}_fb_m{m}"]
            y, z = torch.zeros_like(x), torch.zeros_like(x)
            if M > 0:
                p = self.mul(self.dm[m], self._below(scl, m))
                y, z = y - p, z - 1j * p
            if m < M:
                q = self.mul(self.dp[m], f[f"{scl}_fb_m{m + 1}"])
                y, z = y + q, z - 1j * q
            for k, v in zip(COMPS, (x, y, z)):
                f[f"{vec}{k}_fb_m{m}"] = v

    def rot(self, src, dst):
        """dst = rot(src) / w^2."""
        f, M = self.f, self.M
        for m in range(M + 1):
            bx = torch.zeros_like(f[f"{src}x_fb_m{m}"])
            by = -1j * self.kx * f[f"{src}z_fb_m{m}"]
            bz = 1j * self.kx * f[f"{src}y_fb_m{m}"]
            if M > 0:
                gx, gy, gz = (self._below(src + k, m) for k in COMPS)
                bx = bx + self.mul(self.dm[m], -gz + 1j * gy)
                p = self.mul(self.dm[m], gx)
                by, bz = by - 1j * p, bz + p
            if m < M:
                gx, gy, gz = (f[f"{src}{k}_fb_m{m + 1}"] for k in COMPS)
                bx = bx + self.mul(self.dp[m], gz + 1j * gy)
                p = self.mul(self.dp[m], gx)
                by, bz = by - 1j * p, bz - p
            for k, v in zip(COMPS, (bx, by, bz)):
                f[f"{dst}{k}_fb_m{m}"] = v / self.w[m] ** 2

    def advance(self):
        f, dti = self.f, 1.0 / DZ
        for m in range(self.M + 1):
            w = self.w[m]
            c1, c2, c3 = torch.cos(w * DZ), w * torch.sin(w * DZ), 1 / w ** 2
            for k in COMPS:
                e, g = f[f"E{k}_fb_m{m}"], f[f"G{k}_fb_m{m}"]
                j, n0, n1 = (2 * math.pi * f[f"{n}{k}_fb_m{m}"] for n in ("J", "dN0", "dN1"))
                e1 = c1 * e + c2 * c3 * (g - j) + c3 * (c1 * n0 - n1 - (n0 - n1) * dti * c2 * c3)
                g1 = -c2 * e + c1 * (g - j) + j + c3 * (dti * (1 - c1) * (n0 - n1) - c2 * n0)
                for n, v in (("E", e1), ("G", g1)):
                    v = torch.fft.ifft(v * self.phase.conj(), dim=1)
                    v = v.real.to(v.dtype) if m == 0 else v
                    f[f"{n}{k}_fb_m{m}"] = torch.fft.fft(v * self.damp, dim=1) * self.phase

    def update(self):
        for k in COMPS:
            for m in range(self.M + 1):
                self.f[f"dN0{k}_fb_m{m}"] = self.f[f"dN1{k}_fb_m{m}"]
        self.grad("rho", "dN1")
        self.advance()
        self.rot("G", "B")

    def pulse(self, las):
        """The laser's E and B in real and spectral space."""
        for n in _vec("E", "B", "G"):
            for m in range(self.M + 1):
                z = torch.zeros((self.nr - 1, self.nx), dtype=torch.complex128, device="cuda")
                self.f[f"{n}_fb_m{m}"] = z
        x = self.xmin + self.dx * torch.arange(self.nx, dtype=torch.float64, device="cuda") - las["x0"]
        r = self.rgrid[:, None]
        v = las["a0"] * torch.sin(2 * math.pi * las["k0"] * x) * torch.exp(
            -x ** 2 / las["Lx"] ** 2 - r ** 2 / las["R"] ** 2)
        v = v * (r.abs() < 3.5 * las["R"]) * (x.abs() < 3.5 * las["Lx"])
        e = torch.fft.fft(self.dht[0] @ v[1:], dim=1) * self.phase
        self.f["Ez_fb_m0"] = e  # in focus at x0: no propagation
        self.f["Gz_fb_m0"] = -1j * self.w[0] * torch.where(self.kx >= 0, 1.0, -1.0) * e
        self.rot("G", "B")
        self.backward(_vec("E", "B"))

    # particles
    def cells(self, p):
        r = torch.sqrt(p["y"] ** 2 + p["z"] ** 2)
        fx, fr = (p["x"] - self.xmin) / self.dx, (r - self.rmin) / self.dr
        ix, ir = torch.floor(fx), torch.floor(fr)
        ok = (ix > 0) & (ix < self.nx - 2) & (ir >= 0) & (ir < self.nr - 2)
        return ix.long(), ir.long(), fx - ix, fr - ir, r, ok

    @staticmethod
    def chunks(n, size=1 << 23):
        return [slice(i, min(n, i + size)) for i in range(0, n, size)]

    @staticmethod
    def push(p, dt):
        for k in COMPS:
            p[k] = p[k] + p["p" + k] * (dt * p["g_inv"])

    def deposit(self, p, names, charge, values):
        """Adds charge w values to the planes `names` (CIC, modes 0..M)."""
        nx, nr, M = self.nx, self.nr, self.M
        acc = {(n, q): torch.zeros(nr * nx, dtype=torch.float64, device="cuda")
               for n in names for q in range(1 + 2 * M)}
        for s in self.chunks(p["x"].numel()):
            q = {k: p[k][s] for k in p}
            ix, ir, sx, sr, r, ok = self.cells(q)
            ix, ir, sx, sr, r = (v[ok] for v in (ix, ir, sx, sr, r))
            e1 = torch.complex(q["y"][ok] / r, q["z"][ok] / r)
            val = [v[ok] * q["w"][ok] * charge for v in values(q)]
            for i in (0, 1):
                for j in (0, 1):
                    C = (sr if i else 1 - sr) * (sx if j else 1 - sx)
                    node = (ir + i) * nx + ix + j
                    for n, v in zip(names, val):
                        cv = C * v
                        acc[n, 0].index_add_(0, node, cv)
                        em = e1
                        for m in range(1, M + 1):
                            acc[n, 2 * m - 1].index_add_(0, node, cv * em.real)
                            acc[n, 2 * m].index_add_(0, node, cv * em.imag)
                            em = em * e1
        for n in names:
            for m in range(M + 1):
                v = acc[n, 0] if m == 0 else torch.complex(acc[n, 2 * m - 1], acc[n, 2 * m])
                v = v.reshape(nr, nx)
                self.f[f"{n}_m{m}"] = self.f[f"{n}_m{m}"] + v if f"{n}_m{m}" in self.f else v

    def finish(self, names):
        """Axis treatment and division by the cell volumes."""
        for n in names:
            for m in range(self.M + 1):
                v = self.f[f"{n}_m{m}"]
                v[1] -= v[0]
                self.f[f"{n}_m{m}"] = v * self.dv[:, None]

    def clear(self, names):
        for n in names:
            for m in range(self.M + 1):
                self.f.pop(f"{n}_m{m}", None)

    def currents(self, e):
        self.clear(_vec("J"))
        self.deposit(e, _vec("J"), -1.0, lambda q: [q["p" + k] * q["g_inv"] for k in COMPS])
        self.finish(_vec("J"))

    def charge(self, e, i):
        self.clear(["rho"])
        one = lambda q: [torch.ones_like(q["w"])]
        self.deposit(e, ["rho"], -1.0, one)
        self.deposit(i, ["rho"], 1.0, one)
        self.finish(["rho"])

    def gather(self, p):
        """Gather + Boris push of the particles of the valid cells whose index
        is below their number (the reference's rule)."""
        f, nx, M = self.f, self.nx, self.M
        for n in _vec("E", "B"):
            for m in range(M + 1):
                v = f[f"{n}_m{m}"]
                v[0] = v[1] if m == 0 else -v[1]
        stay = sum(int(self.cells({k: p[k][s] for k in COMPS})[5].sum()) for s in self.chunks(p["x"].numel()))
        h = 0.5 * (2 * math.pi * DZ * -1.0)
        for s in self.chunks(p["x"].numel()):
            q = {k: p[k][s] for k in p}
            ix, ir, sx, sr, r, ok = self.cells(q)
            ok &= torch.arange(s.start, s.stop, device="cuda") < stay
            ix, ir, sx, sr, r = (v[ok] for v in (ix, ir, sx, sr, r))
            g1 = torch.complex(q["y"][ok] / r, -q["z"][ok] / r)
            F = {}
            for n in _vec("E", "B"):
                t = torch.zeros_like(r)
                for i in (0, 1):
                    for j in (0, 1):
                        C = (sr if i else 1 - sr) * (sx if j else 1 - sx)
                        node = (ir + i) * nx + ix + j
                        t += C * f[f"{n}_m0"].reshape(-1)[node]
                        gm = g1
                        for m in range(1, M + 1):
                            t += 2 * C * (f[f"{n}_m{m}"].reshape(-1)[node] * gm).real
                            gm = gm * g1
                F[n] = t
            E, B = (torch.stack([F[n + k] for k in COMPS]) for n in ("E", "B"))
            um = torch.stack([q["p" + k][ok] for k in COMPS]) + h * E
            t = h * B / torch.sqrt(1 + (um ** 2).sum(0))
            sv = 2 * t / (1 + (t ** 2).sum(0))
            u = um + torch.linalg.cross(um + torch.linalg.cross(um, t, dim=0), sv, dim=0) + h * E
            at = ok.nonzero()[:, 0] + s.start
            for k in range(3):
                p["p" + COMPS[k]][at] = u[k]
            p["g_inv"][at] = 1 / torch.sqrt(1 + (u ** 2).sum(0))

    def out(self, names, spectral=False):
        return {f"{n}_m{m}": self.f[f"{n}{'_fb' if spectral else ''}_m{m}"]
                for n in names for m in range(self.M + 1)}


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind == "gradient":
        return None  # a reverse sweep of plain tensor operations needs minutes
    x = _Exact(c)
    if kind == "setup":
        x.pulse(_laser_cfg(c, seed))
        out = x.out(_vec("E", "B"))
        for k, t in (("DHT_m", x.dht), ("DHT_inv_m", x.inv), ("dDHT_plus_m", x.dp), ("dDHT_minus_m", x.dm)):
            out.update({k + str(m): t[m] for m in range(c["m"] + 1)})
        return out
    if kind == "transform":
        x.f.update(_planes(c, ["rho"] + _vec("J"), seed, False))
        x.f.update(_planes(c, _vec("E", "B"), seed + 1, True))
        x.forward(["rho"] + _vec("J"), smooth=True)
        x.backward(_vec("E", "B"))
        return [x.out(["rho"] + _vec("J"), True), x.out(_vec("E", "B"))]
    if kind == "update":
        x.f.update(_planes(c, ["rho"] + _vec("E", "G", "J", "dN1"), seed, True, _AMP))
        x.update()
        return x.out(_vec("E", "G", "B", "dN0", "dN1"), True)
    e = _plasma(c, seed)
    if kind == "gather":
        x.f.update(_planes(c, _vec("E", "B"), seed + 1, False))
        x.gather(e)
        return {k: e[k] for k in ("px", "py", "pz", "g_inv")}
    ions = {k: e[k].clone() for k in ("x", "y", "z", "w")}
    if kind == "deposit":
        x.push(e, 0.5 * DZ)
        x.currents(e)
        x.push(e, 0.5 * DZ)
        x.charge(e, ions)
        return [x.out(_vec("J") + ["rho"]), {k: e[k] for k in COMPS}, {"sort_indx": None, "cell_offset": None}]
    x.pulse(_laser_cfg(c, seed))
    for n in _vec("dN1"):
        for m in range(c["m"] + 1):
            x.f[f"{n}_fb_m{m}"] = torch.zeros((x.nr - 1, x.nx), dtype=torch.complex128, device="cuda")
    for _ in range(c["steps"]):
        x.push(e, 0.5 * DZ)
        x.currents(e)
        x.push(e, 0.5 * DZ)
        x.charge(e, ions)
        x.forward(["rho"] + _vec("J"), smooth=True)
        x.update()
        x.backward(_vec("E", "B"))
        x.gather(e)
    return [x.out(_vec("E", "B", "J") + ["rho"]), {k: e[k] for k in ("x", "y", "z", "px", "py", "pz", "g_inv")}]
