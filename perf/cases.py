"""The calls that a program using this framework makes, with sizes, states and inputs as they occur.

A case is a run of the coupled step through ``Simulation`` (``step``, then the fields and radii that are
saved), or one gradient (``adjoint``).  The medium, source and bubble populations are those of the
benchmark and of the parity tests: water, dx = 0.1 mm, CFL 0.5, a focused continuous wave from the y0
edge, bubbles around the focus; and the reference driver's own ``Sample.txt`` (cylindrical, CFL 0.1,
thermal, mirrors on two sides, one bubble per cell of a box).

A case's keys: ``kind`` ("forward" or "adjoint"); ``setup`` ("focus" or "sample"); ``nx``, ``ny`` cells;
``mixed`` (FP32 fields, else FP64); ``bubbles`` (0: acoustics only) in a box of ``box`` cells;
``radii`` ("uniform" 1..5 um, "lognormal" median 3 um, "clouds": log-normal in 16 Gaussian clouds);
``amp`` source pressure in MPa at ``freq`` MHz; ``elements`` source elements (0: one source);
``start`` steps taken before the state is saved; ``steps`` steps of one pass; ``thermal``.
"""
import importlib
import math

import numpy as np
import torch

brp = importlib.import_module("cuda-rp_amd")
abi = brp.abi

DX = 1.0e-4


def _focal_cells(ny):
    """Focal length in cells: 15 mm, or less where the grid is shorter."""
    return min(150.0, 0.62 * ny / (0.5 * math.sqrt(3.0)))


def _case(name=None, **kw):
    c = dict(kind="forward", setup="focus", nx=256, ny=256, mixed=False, bubbles=0, box=40,
             radii="uniform", amp=0.5, freq=1.0, elements=0, start=0, steps=1, thermal=False)
    c.update(kw)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: one step and its pressure, as a control loop or a test does it
        _case("step_64_fp64", nx=64, ny=64, bubbles=160, box=16, amp=1.0, start=20, steps=1),
        # acoustics alone, to set up a transducer: small, and the largest grid to a save interval
        _case("acoustic_256_fp64", nx=256, ny=256, start=40, steps=20),
        _case("acoustic_4096_mixed", nx=4096, ny=4096, mixed=True, start=40, steps=100),
        # the reference driver's Sample.txt: cylindrical, with the temperature solve, 45 000 bubbles
        _case("sample_300x600_fp64", setup="sample", nx=300, ny=600, thermal=True, start=60, steps=20),
        # a cloud before the wave reaches it (11 sub-steps a bubble, one Picard iteration)
        _case("cloud_256_fp64_early", bubbles=1024, elements=64, start=100, steps=50),
        _case("cloud_2048_mixed_early", nx=2048, ny=2048, mixed=True, bubbles=1 << 20, box=80,
              radii="lognormal", amp=1.5, start=100, steps=20),
        # the same clouds while their bubbles collapse (thousands of sub-steps, 3 to 5 iterations)
        _case("cloud_256_fp64", bubbles=1024, elements=64, start=400, steps=4),
        _case("cloud_2048_fp64", nx=2048, ny=2048, bubbles=1 << 20, box=80, radii="lognormal",
              amp=1.5, start=300, steps=6),
        # odd sizes all through
        _case("ragged_777x1013_mixed", nx=777, ny=1013, mixed=True, bubbles=30011, box=37,
              radii="lognormal", amp=0.9, start=310, steps=7),
        # the headline: 2^22 bubbles in 16 clouds at 3 MPa
        _case("clouds_4096_mixed", nx=4096, ny=4096, mixed=True, bubbles=1 << 22, box=80,
              radii="clouds", amp=3.0, freq=2.0, start=300, steps=16),
        # one gradient: the step differentiated backwards, small in FP64 and at the adjoint workload's size
        _case("adjoint_256_fp64", kind="adjoint", bubbles=1024, elements=64, steps=290),
        _case("adjoint_1024_mixed", kind="adjoint", nx=1024, ny=1024, mixed=True, bubbles=65536,
              elements=64, steps=310),
    ]


def _log_int(r, lo, hi):
    return int(round(math.exp(r.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(("acoustic", "early", "early", "collapse", "collapse", "adjoint", "sample"))
    if family == "sample":
        nx = _log_int(rng, 40, 400)
        return _case(setup="sample", nx=nx, ny=2 * nx + rng.randrange(-7, 8), thermal=rng.random() < 0.7,
                     start=rng.randrange(10, 70), steps=rng.randrange(3, 25))
    if family == "acoustic":
        nx, ny = _log_int(rng, 48, 3000), _log_int(rng, 48, 3000)
        return _case(nx=nx, ny=ny, mixed=rng.random() < 0.5, amp=round(rng.uniform(0.2, 3.0), 3),
                     freq=rng.choice((1.0, 2.0)), elements=rng.choice((0, 16)),
                     start=rng.randrange(5, 60), steps=rng.randrange(1, 100))
    if family == "adjoint":
        nx, ny = _log_int(rng, 80, 400), _log_int(rng, 80, 400)
    else:
        nx, ny = _log_int(rng, 64, 2100), _log_int(rng, 64, 2100)
    f = _focal_cells(ny)
    box = max(4, int(min(rng.uniform(10, 81), 0.5 * nx, 0.5 * f)))
    most = {"early": 1 << 20, "collapse": 1 << 18, "adjoint": 1 << 13}[family]
    c = _case(nx=nx, ny=ny, mixed=rng.random() < 0.5, bubbles=_log_int(rng, 30, most), box=box,
              radii=rng.choice(("uniform", "lognormal", "clouds")), freq=rng.choice((1.0, 2.0)),
              elements=rng.choice((0, 16)))
    if family == "early":
        arrive = int(2 * (f - 0.5 * box))
        start = rng.randrange(5, max(6, min(arrive - 15, 160)))
        c.update(start=start, steps=rng.randrange(1, max(2, min(40, arrive - start - 5))),
                 amp=round(rng.uniform(0.3, 2.0), 3))
    elif family == "collapse":
        # FP32 fields beside few, strongly collapsing bubbles can keep the Picard residual above its
        # threshold; mixed runs in earnest have many bubbles
        mixed = c["mixed"] and c["bubbles"] >= 4096
        c.update(start=int(2 * f) + rng.randrange(0, 60), steps=rng.randrange(1, 7), mixed=mixed,
                 amp=round(rng.uniform(0.4, 1.2 if mixed else 2.0), 3))
    else:
        c.update(kind="adjoint", elements=rng.choice((4, 16)), steps=int(2 * f) - rng.randrange(0, 20),
                 amp=round(rng.uniform(0.2, 0.6), 3))
    return c


# ---- inputs -----------------------------------------------------------------
def _config(c):
    prec = abi.PREC_MIXED if c["mixed"] else abi.PREC_FP64
    if c["setup"] == "sample":
        cfg = abi.default_config()
        lx, ly = c["nx"] * DX, c["ny"] * DX
        cfg.update(grid_x=c["nx"], grid_y=c["ny"], grid_lx=lx, grid_ly=ly, pml_x0=0, pml_x1=1,
                   pml_y0=0, pml_y1=1, pml_grid_number=10, pml_sigma=0.1, pml_order=2, sim_cfl=0.1,
                   sim_order=2, sim_smooth_delta_band=2, tr_amp=1.5e-2, tr_freq=1.0e6,
                   tr_focal_dist=ly * 2.0 / 3.0, tr_box_size=lx, tr_cylindrical=1, tr_on_wave=2,
                   tr_off_wave=0, tr_focused_p=1, bub_enable=1, bub_fg0=1e-7, bub_R0=6.5e-7,
                   bub_P0=0.1e6, bub_T0=293.15, bub_gamma=1.4, bub_sigma=7.2e-2, bub_mu=891.0e-6,
                   bub_rho=1.0e3, bub_K0=26.2e-3, precision=prec, thermal=int(c["thermal"]))
        return cfg
    n = max(c["nx"], c["ny"])
    cfg = abi.water_config(n, npml=32 if n >= 1000 else 16 if n >= 100 else 8, amp_pa=c["amp"] * 1e6,
                           freq=c["freq"] * 1e6, focal_dist=_focal_cells(c["ny"]) * DX,
                           bubbles=c["bubbles"] > 0, precision=prec)
    cfg.update(grid_x=c["nx"], grid_y=c["ny"], grid_lx=c["nx"] * DX, grid_ly=c["ny"] * DX,
               ext_focus_x=0.5 * c["nx"] * DX, thermal=int(c["thermal"]))
    return cfg


def _inputs(c, seed):
    """The population (x, y, R0, fg_in) and the source elements (amplitude, phase) from the seed."""
    r = np.random.default_rng(seed)
    bubbles = source = None
    if c["setup"] == "sample":  # one bubble per cell; the seed varies the source elements below
        source = (22500.0 * (0.8 + 0.4 * r.random(8)), 0.4 * r.random(8))
        return bubbles, source
    n, box = c["bubbles"], c["box"] * DX
    if n:
        fx, fy = 0.5 * c["nx"] * DX, _focal_cells(c["ny"]) * DX * 0.5 * math.sqrt(3.0)
        if c["radii"] == "clouds":
            cx, cy = fx + (r.random(16) - 0.5) * box, fy + (r.random(16) - 0.5) * box
            k = r.integers(0, 16, n)
            s = box / 32.0
            x = np.clip(cx[k] + s * r.standard_normal(n), fx - 0.5 * box, fx + 0.5 * box)
            y = np.clip(cy[k] + s * r.standard_normal(n), fy - 0.5 * box, fy + 0.5 * box)
        else:
            x, y = fx + (r.random(n) - 0.5) * box, fy + (r.random(n) - 0.5) * box
        R0 = 1e-6 + 4e-6 * r.random(n) if c["radii"] == "uniform" else \
            np.exp(np.log(3e-6) + 0.4 * r.standard_normal(n))
        bubbles = (x, y, R0, 1e-6 * c["box"] ** 2 / n)
    ne = c["elements"] or (1 if n == 0 else 0)  # acoustics: the source is all that the seed can vary
    if ne:
        amp = c["amp"] * 1e6 * (0.6 + 0.8 * r.random(ne))
        phase = 2.0 * math.pi * r.random(ne) if c["kind"] == "adjoint" else 0.3 * r.random(ne)
        source = (amp, phase)
    return bubbles, source


def prepare(case, seed):
    """A simulation at the state that the pass starts from, saved in slot 0."""
    bubbles, source = _inputs(case, seed)
    sim = brp.Simulation(_config(case))
    if bubbles is not None:
        x, y, R0, fg_in = bubbles
        sim.set_bubbles(x, y, R0, None, fg_in)
    if source is not None:
        sim.set_source(*source)
    sim.prepare()
    if case["start"]:
        sim.step(case["start"])
    sim.save_state(0)
    ic, jc = int(case["nx"] / 2 + 0.5), int(_focal_cells(case["ny"]) * 0.5 * math.sqrt(3.0) + 0.5)
    half = max(2, min(10, case["box"] // 4))
    return {"sim": sim, "case": case, "box": (ic - half, ic + half - 1, jc - half, jc + half - 1)}


def run(state):
    sim, c = state["sim"], state["case"]
    sim.restore_state(0)
    if c["kind"] == "adjoint":
        r = sim.adjoint(state["box"], c["steps"], max(1, c["steps"] // 10))
        return {k: r[k] for k in ("J", "grad_amp", "grad_phase", "grad_fg0")}
    sim.step(c["steps"])
    out = {"p0": sim.field("p0")}
    if c["bubbles"] or c["setup"] == "sample":
        out["fg"] = sim.field("fg")
        out["R_t"] = sim.bubbles("R_t")
    if c["thermal"]:
        out["T"] = sim.field("T")
    return out


def work(case):
    """Each step reads and writes the five field components and the bubbles' state once; the saved
    fields are written once.  Operations: 40 a cell, and 470 an RP sub-step (11 a bubble before the
    wave arrives; about 20 in each of 4 iterations while bubbles collapse).  A gradient runs every step
    forwards and backwards."""
    cells = case["nx"] * case["ny"]
    nb, word = case["bubbles"], 4 if case["mixed"] else 8
    if case["setup"] == "sample":
        nb = cells // 4
    early = case["start"] + case["steps"] < 2 * _focal_cells(case["ny"]) or case["setup"] == "sample"
    passes = 2 if case["kind"] == "adjoint" else 1
    step_bytes = cells * (10 * word + (16 if case["thermal"] else 0)) + nb * 208
    step_flops = cells * 40 + nb * 470 * (11 if early else 80)
    return {"bytes": passes * case["steps"] * step_bytes + 8 * (cells * (1 + (nb > 0)) + nb),
            "flops": passes * case["steps"] * step_flops}


# ---- the same numbers in 64 bits, from the equations ------------------------
def exact(case, seed):
    """The run from rest to the end of the pass by the model's equations in float64.  None for
    collapsing bubbles (thousands of sequential sub-steps) and for gradients."""
    early = case["setup"] == "sample" or not case["bubbles"] or \
        case["start"] + case["steps"] < 2 * (_focal_cells(case["ny"]) - 0.5 * case["box"])
    if case["kind"] == "adjoint" or not early:
        return None
    nb = case["bubbles"] or (case["nx"] * case["ny"] // 4 if case["setup"] == "sample" else 0)
    if (case["start"] + case["steps"]) * (nb / 2e7 + case["nx"] * case["ny"] / 1e9 + (0.06 if nb else 0.003)) > 20:
        return None
    m = _Model(case, seed)
    for _ in range(case["start"] + case["steps"]):
        m.step()
    out = {"p0": m.p0[1:, 1:].cpu()}
    if m.nb:
        out["fg"], out["R_t"] = m.fg[1:, 1:].cpu(), m.R_t.cpu()
    if case["thermal"]:
        out["T"] = m.T[1:, 1:].cpu()
    return out


def _cdiv(a, b):
    d = b[0] * b[0] + b[1] * b[1]
    return (a[0] * b[0] + a[1] * b[1]) / d, (a[1] * b[0] - a[0] * b[1]) / d


def _cmul(a, b):
    return a[0] * b[0] - a[1] * b[1], a[1] * b[0] + a[0] * b[1]


class _Model:
    """The coupled step on float64 tensors.  Grid arrays hold rows j = -1..M+1, columns i = -1..N+1;
    element (i, j) is [j + 1, i + 1]."""

    def __init__(self, case, seed):
        self.c = c = _config(case)
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.N, self.M = N, M = c.grid_x, c.grid_y
        self.dx, self.dy = c.grid_lx / N, c.grid_ly / M
        self.rho, self.cs, self.P_inf, self.T_inf = 1000.0, 1500.0, 0.1e6, 293.15
        self.dt = c.sim_cfl * min(self.dx, self.dy) / self.cs
        self.fx = c.ext_focus_x if c.ext_focus_x_set else 0.0
        self.fy = c.tr_focal_dist * 0.5 * math.sqrt(3.0)
        self.fdist = self.fy / 0.5 / math.sqrt(3.0)
        self.omega = 2.0 * math.pi * c.tr_freq
        z = lambda v=0.0: torch.full((M + 3, N + 3), v, dtype=torch.float64, device=self.dev)  # noqa: E731
        self.p0, self.px, self.py, self.vx, self.vy = z(), z(), z(), z(), z()
        self.fg, self.fgn, self.fgm = z(), z(), z()
        self.rho_m = z(self.rho)
        if c.thermal:
            self.T, self.C_pm = z(), self._heat_capacity(z())
        self.nx_s, self.ny_s, self.mx_s, self.my_s = self._pml()
        self.t, self.tx, self.nb = 0.0, 0.0, 0
        bubbles, source = _inputs(case, seed)
        self.source = None if source is None else tuple(self._t(v) for v in source)
        if c.bub_enable:
            self._place(bubbles)
            self.fg = self._scatter(self.pi43 * self.n_B * self.R_t ** 3)
            self.fgn, self.fgm = self.fg.clone(), self.fg.clone()

    def _t(self, v):
        return torch.as_tensor(np.asarray(v, dtype=np.float64), device=self.dev)

    def _pml(self):
        c, n = self.c, self.c.pml_grid_number

        def profile(size, d, lo, hi, first, half):
            out = np.zeros(size + 3)
            smax = -math.log(c.pml_sigma) * 0.5 * (c.pml_order + 1.0) / (d * n)
            for i in range(first, size + 1):
                if lo and i <= n - (1 - first):
                    out[i + 1] = smax * ((n - i + first - half) / n) ** c.pml_order
                if hi and i >= size - n + 1:
                    out[i + 1] = smax * ((i - size + n - half) / n) ** c.pml_order
            return out
        x = lambda first, half: profile(self.N, self.dx, c.pml_x0, c.pml_x1, first, half)  # noqa: E731
        y = lambda first, half: profile(self.M, self.dy, c.pml_y0, c.pml_y1, first, half)  # noqa: E731
        return self._t(x(0, 0.0)), self._t(y(0, 0.0))[:, None], self._t(x(1, 0.5)), self._t(y(1, 0.5))[:, None]

    def _place(self, bubbles):
        c = self.c
        if bubbles is None:
            i, j = np.meshgrid(np.arange(1, self.N + 1), np.arange(1, self.M + 1), indexing="ij")
            x, y = (i - 0.5) * self.dx, (j - 0.5) * self.dy
            keep = (np.abs(x - self.fx) < 0.5 * c.tr_box_size) & (np.abs(y - self.fy) < 0.5 * c.tr_box_size)
            x, y = x[keep], y[keep]
            R0, fg_in = np.full(x.shape, c.bub_R0), c.bub_fg0
        else:
            x, y, R0, fg_in = bubbles
        self.x, self.y, self.R0 = self._t(x), self._t(y), self._t(R0)
        self.nb = len(x)
        self.pi43 = math.pi * 4.0 / 3.0
        self.PG0 = c.bub_P0 + 2.0 * c.bub_sigma / self.R0
        self.ca = c.bub_gamma * self.PG0 * self.R0 ** 3 / (2.0 * (c.bub_gamma - 1.0) * c.bub_T0 * c.bub_K0)
        self.n_B = fg_in * self.dx * self.dy * (self.x if c.tr_cylindrical else 1.0) / (self.pi43 * self.R0 ** 3)
        zero = torch.zeros_like(self.x)
        self.rp = [self.R0.clone(), self.R0.clone(), zero, self.PG0.clone(),
                   torch.full_like(self.x, 0.1 * self.dt), zero]  # R, previous R, dR/dt, PG, dt, rest
        self.R_t, self.PLm, self.PLn, self.PLp, self.Q_B = self.R0.clone(), zero, zero, zero, zero

    # -- bubbles and grid
    def _stencil(self, cx, cy):
        """Weights and flat places of each bubble's cells: columns from floor(x/dx + cx), rows likewise."""
        w = self.c.sim_smooth_delta_band
        sx, sy = (-(w // 2) + (1 if cc == 0.5 else 0) for cc in (cx, cy))
        bx, by = torch.floor(self.x / self.dx + cx).long(), torch.floor(self.y / self.dy + cy).long()
        for a in range(w):
            i = bx + sx + a
            Dx = (1.0 + torch.cos(2.0 * math.pi / w / self.dx * ((i.double() - 0.5) * self.dx - self.x))) / w
            for b in range(w):
                j = by + sy + b
                Dy = (1.0 + torch.cos(2.0 * math.pi / w / self.dy * ((j.double() - 0.5) * self.dy - self.y))) / w
                ok = (i >= (-1 if cx == 1.0 else 0)) & (i <= self.N + 1) & (j >= (-1 if cy == 1.0 else 0)) & (j <= self.M + 1)
                at = ((j + 1) * (self.N + 3) + i + 1).clamp(0, (self.N + 3) * (self.M + 3) - 1)
                yield at, torch.where(ok, Dx * Dy, torch.zeros_like(Dx))

    def _gather(self, f, cx=0.5, cy=0.5):
        return sum(f.reshape(-1)[at] * w for at, w in self._stencil(cx, cy))

    def _scatter(self, v, fold=True):
        v = v / (self.dx * self.dy)
        if self.c.tr_cylindrical:
            v = v / self.x
        f = torch.zeros((self.M + 3) * (self.N + 3), dtype=torch.float64, device=self.dev)
        for at, w in self._stencil(0.5, 0.5):
            f.index_add_(0, at, v * w)
        f = f.reshape(self.M + 3, self.N + 3)
        if fold and self.c.tr_cylindrical:
            f[:, 1] += f[:, 2]
            f[:, 2] = f[:, 1]
        return f

    # -- one step
    def step(self):
        c, N, M = self.c, self.N, self.M
        s = self.t
        self.t = self.t + self.dt + self.tx
        self.tx = self.dt + self.tx - (self.t - s)
        pn = (self.px, self.py)
        self.fgm, self.fgn, self.fg = self.fgn, self.fg, 3.0 * self.fg - 3.0 * self.fgn + self.fgm
        self._velocity()
        if self.nb:
            self.PLm, self.PLn = self.PLn, self.PLp
            vx, vy = self._gather(self.vx, 1.0, 0.5), self._gather(self.vy, 0.5, 1.0)
            self.x, self.y = self.x + vx * self.dt, self.y + vy * self.dt
        res = self._pressure(pn)
        start = self.rp if self.nb else None
        while self.nb and res > float(np.float32(1.0e-7)):
            self.PLp = self._gather(self.p0)
            self.rp = self._radii(start)
            self.fg = self._scatter(self.pi43 * self.n_B * self.R_t ** 3)
            res = self._pressure(pn)
        if c.thermal:
            self._temperature(pn)
            self.C_pm = self._heat_capacity(self.T)
        self.rho_m = (1.0 - self.fg) * self.rho

    def _velocity(self):
        c, N, M, p = self.c, self.N, self.M, self.p0
        vx, vy = self.vx, self.vy
        s = 0.5 * self.dt * self.cs
        at = (slice(2, M + 2), slice(1, N + 2))       # rows 1..M, nodes 0..N
        to = (slice(2, M + 2), slice(2, N + 3))
        sx = s * self.nx_s[1:N + 2]
        vx[at] = (vx[at] * (1.0 - sx) - self.dt / (0.5 * (self.rho_m[at] + self.rho_m[to])) * (p[to] - p[at]) / self.dx) / (1.0 + sx)
        at = (slice(1, M + 2), slice(2, N + 2))       # nodes 0..M, columns 1..N
        to = (slice(2, M + 3), slice(2, N + 2))
        sy = s * self.ny_s[1:M + 2]
        vy[at] = (vy[at] * (1.0 - sy) - self.dt / (0.5 * (self.rho_m[at] + self.rho_m[to])) * (p[to] - p[at]) / self.dx) / (1.0 + sy)
        # walls and ghosts, in the reference's order
        if not c.pml_x0:
            vx[2:M + 2, 0], vx[2:M + 2, 1] = vx[2:M + 2, 2], 0.0
        if not c.pml_x1:
            vx[2:M + 2, N + 2], vx[2:M + 2, N + 1] = -vx[2:M + 2, N], 0.0
        vx[1], vx[M + 2] = vx[2], vx[M + 1]
        if not c.pml_y0:
            if not c.tr_plane_p and not c.tr_focused_p:
                vy[1, 2:N + 2] = 0.0
            vy[0, 2:N + 2] = vy[1, 2:N + 2]
        if not c.pml_y1:
            vy[M + 1, 2:N + 2] = 0.0
            vy[M + 2, 2:N + 2] = vy[M, 2:N + 2]
        corner = vy[N + 1, N + 1].clone() if N <= M + 1 else 0.0
        vy[:, 1] = vy[:, 2]
        vy[:, N + 2] = corner

    def _pressure(self, pn):
        c, N, M = self.c, self.N, self.M
        q = (slice(2, M + 2), slice(2, N + 2))
        vx, vy = self.vx, self.vy
        if c.tr_cylindrical:
            xu = torch.arange(-1, N + 2, dtype=torch.float64, device=self.dev) * self.dx
            mid = self.dx * (torch.arange(1, N + 1, dtype=torch.float64, device=self.dev) - 0.5)
            s1x = (-xu[1:N + 1] * vx[2:M + 2, 1:N + 1] + xu[2:N + 2] * vx[q]) / self.dx / mid
        else:
            s1x = (vx[q] - vx[2:M + 2, 1:N + 1]) / self.dx
        s1y = (vy[q] - vy[1:M + 1, 2:N + 2]) / self.dy
        s3 = self.dt * self.rho * self.cs * self.cs
        s5 = -(self.fg[q] - self.fgn[q]) / self.dt / (1.0 - 0.5 * (self.fg[q] + self.fgn[q]))
        sx, sy = 0.5 * self.dt * self.cs * self.mx_s[2:N + 2], 0.5 * self.dt * self.cs * self.my_s[2:M + 2]
        self.px, self.py = pn[0].clone(), pn[1].clone()
        self.px[q] = pn[0][q] * (1.0 - sx) - s3 * (s1x + 0.5 * s5) / (1.0 + sx)
        self.py[q] = pn[1][q] * (1.0 - sy) - s3 * (s1y + 0.5 * s5) / (1.0 + sy)
        new = self.px[q] + self.py[q]
        res = float((self.p0[q] - new).abs().max()) / self.P_inf
        p = self.p0
        p[q] = new
        if not c.pml_y0:
            p[1, 2:N + 2] = p[2, 2:N + 2]
        if not c.pml_y0 or c.ext_source_in_pml:
            p[1, 2:N + 2] = self._source()
        if not c.pml_y1:
            for j in (N, N + 1):
                if j <= M + 1 and 0 <= 2 * M + 1 - j <= M + 1:
                    p[j + 1, 2:N + 2] = p[2 * M + 2 - j, 2:N + 2]
        if not c.pml_x0:
            p[1:, 1] = p[1:, 2]
        if not c.pml_x1:
            p[1:, N + 2] = p[1:, N + 1]
        return res

    def _source(self):
        c = self.c
        xm = (torch.arange(1, self.N + 1, dtype=torch.float64, device=self.dev) - 0.5) * self.dx
        r = torch.sqrt((self.fx - xm) ** 2 + (self.fy + 0.5 * self.dy) ** 2)
        on = r <= self.fdist
        t = torch.clamp(self.t - (self.fdist - r) / self.cs, min=0.0)
        t = torch.fmod(t, (c.tr_on_wave + c.tr_off_wave) / c.tr_freq)
        amp, phase = torch.full_like(xm, self.rho * self.cs * c.tr_amp), torch.zeros_like(xm)
        if self.source is not None and bool(on.any()):
            k = torch.nonzero(on).reshape(-1)
            e = ((torch.arange(self.N, device=self.dev) - k[0]) * len(self.source[0]) // (k[-1] - k[0] + 1)).clamp(0, len(self.source[0]) - 1)
            amp, phase = self.source[0][e], self.source[1][e]
        return torch.where(on & (t < c.tr_on_wave / c.tr_freq), amp * torch.sin(self.omega * t + phase), 0.0)

    def _upsilon(self, s):
        """(a coth a - 1) / a^2 for a = s (1 + i): closed form, or its series for small |a|; and Lp / R."""
        x, y = torch.tanh(s), torch.tan(s)
        one = torch.ones_like(s)
        ac = _cmul((s, s), _cdiv((one, x * y), (x, y)))
        g = (ac[0] - 1.0, ac[1])
        q = 2.0 * s * s                                # a^2 = i q
        U = (g[1] / q, -g[0] / q)
        W = _cdiv((-3.0 * g[0], q - 3.0 * g[1]), (-q * g[1], q * g[0]))
        iq = lambda v: (-q * v[1], q * v[0])           # noqa: E731
        Us = iq((2.0 / 945.0 * one, -q / 4725.0))
        Us = iq((Us[0] - 1.0 / 45.0, Us[1]))
        Us = (Us[0] + 1.0 / 3.0, Us[1])
        Ws = iq((2.0 / 7875.0 * one, -q * 37.0 / 3031875.0))
        Ws = iq((Ws[0] - 1.0 / 175.0, Ws[1]))
        Ws = (Ws[0] + 1.0 / 5.0, Ws[1])
        big = math.sqrt(2.0) * s > 0.1
        pick = lambda u, v: tuple(torch.where(big, a, b) for a, b in zip(u, v))  # noqa: E731
        return pick(U, Us), pick(W, Ws)

    def _radii(self, start):
        """Every bubble's Rayleigh-Plesset integration over the step, from its state at the step's start."""
        c, eps, dt_mix = self.c, 2.22044604925031308e-16, self.dt
        out = [v.clone() for v in start]
        R_t, Q = self.R_t.clone(), self.Q_B.clone()
        k = torch.arange(self.nb, device=self.dev)
        R, Rn, d1, PG, dt, rest = (v.clone() for v in start)
        remain, time = rest + dt_mix, -rest
        P0, P1 = self.PLn + c.bub_P0, 0.5 * (self.PLp - self.PLm) / dt_mix
        P2 = 0.5 * (self.PLp + self.PLm - 2.0 * self.PLn) / (dt_mix * dt_mix)
        heat = torch.zeros_like(R)
        R0, PG0, ca, rest0 = self.R0, self.PG0, self.ca, rest
        gam, mu, rho, sig = c.bub_gamma, c.bub_mu, c.bub_rho, c.bub_sigma
        while len(k):
            Rm, Rn, PGn = Rn, R, PG
            PL = P2 * time * time + P1 * time + P0
            acc = (PGn - PL - 2.0 * sig / Rn - 4.0 * mu / Rn * d1) / rho - 1.5 * d1 * d1
            dtm = dt
            dt = torch.clamp(1.01 * dtm, max=0.1 * dt_mix)
            dt = torch.where(d1.abs() > eps, torch.minimum(dt, 0.01 * Rn / d1.abs()), dt)
            dt = torch.where(acc.abs() > eps, torch.minimum(dt, 0.1 * Rn / torch.sqrt(acc.abs())), dt)
            at = lambda h: (1.0 + h / dtm) * Rn - h / dtm * Rm + (h / Rn) * (0.5 * (h + dtm) * acc)  # noqa: E731
            R = at(dt)
            d1 = (dtm * dtm * R + (dt * dt - dtm * dtm) * Rn - dt * dt * Rm) / (dtm * dt * (dtm + dt)) + dt / Rn * acc
            last = dt >= remain
            Rt = torch.where(last, at(remain), R)
            remain = remain - torch.where(last, remain, dt)
            time = time + dt
            # solveOmegaN: three fixed-point iterations, then Lp
            A, v1, c3 = 3.0 * gam * PG0 * rho * (R0 / Rn) ** 3, -2.0 * sig * rho / Rn, 4.0 / (Rn * Rn)
            eta = A + v1 - mu * mu * c3
            om = torch.sqrt(torch.clamp(eta, min=1e-6 * eps)) / (rho * Rn)
            for _ in range(3):
                U, _w = self._upsilon(torch.sqrt(ca / Rn * om))
                V = _cdiv((torch.ones_like(om), torch.zeros_like(om)), (1.0 + 3.0 * (gam - 1.0) * U[0], 3.0 * (gam - 1.0) * U[1]))
                m = mu + 3.0 * gam * V[1] * PG0 * (R0 / Rn) ** 3 / (4.0 * om)
                eta = V[0] * A + v1 - m * m * c3
                om = torch.sqrt(torch.clamp(eta, min=1e-6 * eps)) / (rho * Rn)
            _u, W = self._upsilon(torch.sqrt(ca / Rn * om))
            L2 = (W[0] * W[0] + W[1] * W[1]) * Rn
            LR, LI = W[0] / L2, W[1] / L2
            Rb = 0.5 * (R + Rn)
            c0 = dt * 3.0 * (gam - 1.0) * c.bub_K0 * c.bub_T0 / (Rb * PG0)
            k3 = 1.5 * gam * (R - Rn) / Rb + c0 * LR * 0.5 * (Rb / R0) ** 3
            k1 = 1.0 + k3 - c0 * LI / (om * dt) * (R / R0) ** 3
            k2 = 1.0 - k3 - c0 * LI / (om * dt) * (Rn / R0) ** 3
            PG = (k2 * PGn + c0 * LR * PG0) / k1
            if c.thermal:
                E = c.bub_T0 / (PG0 * R0 ** 3)
                dT = LR * E * (PG0 * R0 ** 3 - 0.5 * (PG + PGn) * Rb ** 3) + LI * E * (PG * R ** 3 - PGn * Rn ** 3) / (om * dt)
                heat = heat - 4.0 * math.pi * R * R * c.bub_K0 * dT * dt + 16.0 * math.pi * mu * R * d1 * d1 * dt
            done = ~(remain > 0.0)
            if bool(done.any()):
                i, go = k[done], ~done
                for o, v in zip(out, (R, Rn, d1, PG, dt, remain)):
                    o[i] = v[done]
                R_t[i] = Rt[done]
                Q[i] = heat[done] / (dt_mix - remain[done] + rest0[done])
                k = k[go]
                R, Rn, d1, PG, dt, remain, time, heat, P0, P1, P2, R0, PG0, ca, rest0 = (
                    v[go] for v in (R, Rn, d1, PG, dt, remain, time, heat, P0, P1, P2, R0, PG0, ca, rest0))
        self.R_t, self.Q_B = R_t, Q
        return out

    # -- temperature (the property fits' literals are single precision, as the model's)
    def _heat_capacity(self, T):
        f = lambda v: float(np.float32(v))  # noqa: E731
        T = T + self.T_inf
        return (917.5 - f(10.1016) * T + f(0.0454134) * T ** 2 - 9.07517e-5 * T ** 3 + f(6.80700e-8) * T ** 4) / f(18.0e-3)

    def _temperature(self, pn):
        c, N, M, T = self.c, self.N, self.M, self.T
        f = lambda v: float(np.float32(v))  # noqa: E731
        Ta = T + self.T_inf
        km = (0.76760 + f(7.5390e-3) * Ta - f(9.8250e-6) * Ta * Ta) * (1.0 - 3.0 * self.fg / (2.0 + self.fg))
        heat = self._scatter(self.n_B * self.Q_B, fold=False) if self.nb else torch.zeros_like(T)
        w, e, d = km[1:, 1:-1], km[1:, 2:], T[1:, 2:] - T[1:, 1:-1]   # x faces 0..N of rows 0..M+1
        Ex = 2.0 * w * e / (w + e) * d / self.dx
        w, e, d = km[1:-1, 1:], km[2:, 1:], T[2:, 1:] - T[1:-1, 1:]
        Ey = 2.0 * w * e / (w + e) * d / self.dy
        q = (slice(2, M + 2), slice(2, N + 2))
        dp = (self.px[q] + self.py[q] - pn[0][q] - pn[1][q]) / self.dt
        ac = 2.0 * 0.22 * 0.115129255 / (self.rho * self.cs * self.omega ** 2) * dp * dp
        div = (Ex[1:M + 1, 1:] - Ex[1:M + 1, :-1]) / self.dx + (Ey[1:, 1:N + 1] - Ey[:-1, 1:N + 1]) / self.dy
        T[q] += self.dt * (div + heat[q] + ac) / (self.rho_m[q] * self.C_pm[q])
        if not c.pml_x0:
            T[2:M + 2, 1] = T[2:M + 2, 2]
        if not c.pml_x1:
            T[1:, N + 2] = T[1:, N + 1]
        if not c.pml_y0:
            T[1, 1:] = T[2, 1:]
        if not c.pml_y1:
            T[M + 1, 1:] = T[M + 2, 1:]
            T[M + 2, 1:] = T[M + 1, 1:]
