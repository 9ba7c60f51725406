"""The work a user of the step engine has it do, as timed cases.

A case is one of four kinds, each through the public entry points of
``lesamd``:

* ``run``: a domain is created from its set-up, advanced ``steps`` whole steps
  and its fields are read back -- what the serving runtime does for one
  request, and what a simulation program does between two outputs.  Options:
  replay from a graph, masks and cn1 given as arrays (``dense``), the time
  statistics of every step (``stats``), inflow planes read per step
  (``planes``), the FP64 defect-correction press (``dc``);
* ``step``: a program that keeps its domain and reads u, v, w and p after
  every step (the smallest calls: launches and latency count);
* ``batch``: several domains of different sizes advanced together;
* ``stages``: the seven reference-signature calls per step on host arrays, as
  the reference's time loop makes them, then the arrays synchronised.

Sizes are those of the named workloads, of the served mix and of the tests,
and ragged ones between them.  ``exact`` is the same time step written in
64-bit torch from the reference's formulas.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mpi-les_amd"))

from lesamd import api, layout, setup_gen  # noqa: E402

FIELDS = ("u", "v", "w", "p")
DEFAULTS = dict(kind="run", dx=4.0, dt=0.05, ustar=0.4, nmaxp=50, omega=1.0, graph=True, dense=False, stats=False,
                planes=False, dc=False)


def _case(name, im, jm, km, steps, **kw):
    return dict(DEFAULTS, name=name, im=im, jm=jm, km=km, steps=steps, **kw)


def listed():
    return [
        # a small domain coupled to another program: one step, fields read, again
        _case("step-24x20x16", 24, 20, 16, 1, kind="step", dt=0.02),
        # a small run without graph replay, the default of a new domain
        _case("run-eager-48x40x24", 48, 40, 24, 100, graph=False),
        # the smallest served class
        _case("run-96x96x64", 96, 96, 64, 100),
        # the reference's own grid
        _case("run-150x150x90", 150, 150, 90, 60),
        # a grid cut out of a city map: odd in every direction
        _case("run-ragged-203x117x61", 203, 117, 61, 60),
        # the benchmark workload
        _case("run-300x300x90", 300, 300, 90, 50),
        # a fine grid (2 m) with the SOR cap of the fine workloads
        _case("run-512x512x128", 512, 512, 128, 24, dx=2.0, dt=0.02, nmaxp=100),
        # the largest workload
        _case("run-1024x1024x128", 1024, 1024, 128, 8, dx=2.0, dt=0.02, nmaxp=100),
        # set-up given as arrays, file-driven inflow and time statistics
        _case("run-stats-160x128x64", 160, 128, 64, 40, dt=0.02, dense=True, stats=True, planes=True),
        # the precision variant of the press
        _case("run-dc-256x256x64", 256, 256, 64, 16, dx=2.0, dt=0.02, nmaxp=100, dc=True),
        # small served domains in one batch
        _case("batch-9-of-96..160", 160, 160, 64, 40, kind="batch"),
        # the drop-in calls of the reference's time loop
        _case("stages-128x96x64", 128, 96, 64, 40, kind="stages", dense=True),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run"] * 7 + ["step", "batch", "stages"])
    im, jm, km = _log_uniform(rng, 20, 640), _log_uniform(rng, 20, 640), rng.choice([16, 24, 37, 48, 64, 90, 96, 105, 128])
    if rng.random() < 0.5:  # grids are mostly even across the wind
        jm += jm % 2
    steps = rng.choice([12, 20, 30, 40, 60])
    if im * jm * km > 12e6:
        steps = min(steps, 12)
    fine = rng.random() < 0.3
    c = dict(DEFAULTS, kind=kind, im=im, jm=jm, km=km, steps=steps, ustar=rng.choice([0.2, 0.25, 0.3, 0.35, 0.4]),
             dx=2.0 if fine else 4.0, dt=0.02 if fine else rng.choice([0.02, 0.05]), nmaxp=100 if fine else 50)
    if kind == "run":
        c["graph"] = rng.random() < 0.8
        if im * jm * km < 6e6:
            c["dense"] = rng.random() < 0.3
            c["stats"] = rng.random() < 0.25
            c["planes"] = rng.random() < 0.25
            if c["planes"]:
                c["dt"] = 0.02
            c["dc"] = rng.random() < 0.15
            if not c["dc"]:
                c["omega"] = rng.choice([1.0, 1.0, 1.0, 1.5])
    elif kind == "step":
        c.update(im=rng.randint(16, 32), jm=rng.randint(16, 32), km=rng.randint(8, 16), steps=1, dt=0.02, nmaxp=50, dx=4.0)
    elif kind == "batch":
        c.update(im=min(im, 192), jm=min(jm, 192) // 2 * 2, km=min(km, 64), steps=min(steps, 20))
    elif kind == "stages":
        c.update(im=min(im, 200), jm=min(jm, 200), km=min(km, 96), dense=True)
    return c


# ------------------------------------------------------------------ the cases
def _workload(c, seed, im, jm, km):
    city = setup_gen.CityParams(4, 2, 0.8, 6.0, 0.5) if min(im, jm) < 64 else (
        setup_gen.CityParams(8, 2, 1.0, 16.0, 0.5) if c["dx"] >= 4 else setup_gen.CityParams(10, 3, 0.6, 20.0, 0.6))
    return setup_gen.Workload(f"case-{im}x{jm}x{km}", im, jm, km, dx=c["dx"], dy=c["dx"], city=city, ustar=c["ustar"],
                              z0=0.1, dt=c["dt"], nsteps=c["steps"], nmaxp=c["nmaxp"], pjuge=1e-6, omega=c["omega"],
                              seed=seed)


def _extents(c):
    """The domains of a case (one, or the batch's nine)."""
    if c["kind"] != "batch":
        return [(c["im"], c["jm"], c["km"])]
    side = lambda n, q: max(16, n - q * (n // 5))  # noqa: E731
    return [(side(c["im"], a), side(c["jm"], b) // 2 * 2, c["km"]) for a in range(3) for b in range(3)]


def _setups(c, seed):
    return [setup_gen.build(_workload(c, seed + 97 * q, *e), dense=c["dense"]) for q, e in enumerate(_extents(c))]


def _planes(c, seed):
    """Inflow planes of every step: the profile with a moving perturbation."""
    rng = np.random.default_rng(seed + 31)
    jm, km = c["jm"], c["km"]
    base = setup_gen.inflow_profile(_workload(c, seed, c["im"], jm, km), setup_gen.grid_metrics(
        _workload(c, seed, c["im"], jm, km)))
    amp = rng.uniform(0.01, 0.03, size=3)
    j = np.arange(jm)[:, None]
    out = []
    for n in range(c["steps"]):
        wave = np.sin(2 * np.pi * (j + n) / jm)
        out.append([np.asfortranarray((base * (1 + amp[0] * wave)).astype(np.float32)),
                    np.asfortranarray((base * amp[1] * wave).astype(np.float32)),
                    np.asfortranarray((base * amp[2] * wave).astype(np.float32))])
    return out


def _domain(c, setup):
    d = api.Domain(setup)
    d.set_graph(c["graph"])
    if c["dc"]:
        d.set_press_mode(1, outer=4, inner=c["nmaxp"] // 4)
    return d


def prepare(case, seed):
    c = dict(DEFAULTS, **case)
    s = dict(case=c, setups=_setups(c, seed), n=0)
    if c["kind"] in ("run", "step"):
        d = _domain(c, s["setups"][0])
        d.autotune()  # timed once per grid shape and process, as at a server's start
        if c["kind"] == "step":
            s["dom"] = d
        else:
            d.close()
        if c["planes"]:
            s["planes"] = _planes(c, seed)
    elif c["kind"] == "stages":
        s["arrays"] = _host_arrays(s["setups"][0])
        s["start"] = {n: a.copy() for n, a in s["arrays"].items() if n in layout.STEP_FIELDS}
    return s


def _host_arrays(setup):
    """The reference program's arrays: zero fields and the set-up."""
    w = setup.workload
    a = {n: layout.new_field(n, w.im, w.jm, w.km) for n in layout.STEP_FIELDS}
    for n, x in setup.masks.items():
        a[n] = np.asfortranarray(x.astype(np.float32))
    for n, x in setup.metrics.items():
        a[n] = np.ascontiguousarray(x.astype(np.float32))
    for n in ("cn2l", "cn2s", "cn3l", "cn3s", "cn4l", "cn4s"):
        a[n] = np.ascontiguousarray(setup.coeffs[n].astype(np.float32))
    a["cn1"] = np.asfortranarray(setup.coeffs["cn1"].astype(np.float32))
    a["delx1"] = layout.new_metric("delx1", w.im, w.jm, w.km)
    return a


def run(state):
    c = state["case"]
    return {"run": _run, "step": _run_step, "batch": _run_batch, "stages": _run_stages}[c["kind"]](state, c)


def _run(state, c):
    d = _domain(c, state["setups"][0])
    d.autotune()
    nmax = c["steps"]
    if c["stats"] or c["planes"]:
        for n in range(1, nmax + 1):
            if c["planes"]:
                d.set_inflow(*state["planes"][n - 1])
            d.step(n, nmax)
            if c["stats"]:
                d.aveflow(n, 2, nmax)
    else:
        d.run(1, nmax, nmax)
    out = {n: d.download(n) for n in FIELDS}
    if c["stats"]:
        out.update({n: d.download(n) for n in layout.AVE_FIELDS})
    d.close()
    return out


def _run_step(state, c):
    d = state["dom"]
    state["n"] += 1
    d.step(state["n"], 1 << 30)
    return {n: d.download(n) for n in FIELDS}


def _run_batch(state, c):
    doms = [_domain(c, s) for s in state["setups"]]
    b = api.Batch(doms, graph=c["graph"])
    for n in range(1, c["steps"] + 1):
        b.step([n] * len(doms), [c["steps"]] * len(doms))
    b.synchronize()
    out = [{n: d.download(n) for n in FIELDS} for d in doms]
    b.close()
    for d in doms:
        d.close()
    return out


def _run_stages(state, c):
    w = state["setups"][0].workload
    a = state["arrays"]
    for n, x in state["start"].items():
        a[n][...] = x
    for x in a.values():
        api.mark_host_dirty(x)
    api.press_config(w.nmaxp, w.pjuge, w.omega)
    api.set_inflow(w.im, w.jm, w.km, state["setups"][0].inflow)
    sc = dict(km=w.km, jm=w.jm, im=w.im, ro=1.1763, dt=w.dt, alpha=-10.0, beta=-1.0, vn=float(setup_gen.VN),
              nmax=c["steps"])
    calls = [(s, {x: sc[x] if x in sc else a[x] for x in api.SIGNATURES[s] if x != "n"}) for s in api.STAGES]
    for n in range(1, c["steps"] + 1):
        for s, args in calls:
            if "n" in api.SIGNATURES[s]:
                args["n"] = n
            api.call(s, **args)
    for n in FIELDS:
        api.sync_host(a[n])
    return {n: a[n] for n in FIELDS}


def work(case):
    """One pass: per step every carried field read and written once (u, v, w,
    p, f, g, h, fold, gold, hold, usum, vsum, wsum) and the step's other
    results written (sm, diu1..9, rhs), 148 B per cell, and the statistics
    100 B; 17 operations per cell and SOR iteration and about 500 for the
    stencils; the fields read back once."""
    c = dict(DEFAULTS, **case)
    n = sum(a * b * k for a, b, k in _extents(c))
    per = 148 + (100 if c["stats"] else 0)
    return {"bytes": float(n * (c["steps"] * per + 16)), "flops": float(n * c["steps"] * (17 * c["nmaxp"] + 500))}


# ------------------------------------------------------------- 64-bit results
def exact(case, seed):
    c = dict(DEFAULTS, **case)
    cells = sum(a * b * k for a, b, k in _extents(c))
    if cells * c["steps"] * (c["nmaxp"] + 10) > 8.5e10 or cells > 40e6:
        return None  # over about 20 seconds
    outs = []
    for s in _setups(c, seed):
        r = _Exact(c, s)
        planes = _planes(c, seed) if c["planes"] else None
        for n in range(1, c["steps"] + 1):
            r.step(n, planes[n - 1] if planes else None)
            if c["stats"]:
                r.aveflow(n, 2, c["steps"])
        outs.append(r.results())
        del r
    return outs if c["kind"] == "batch" else outs[0]


class _Exact:
    """The time step in 64 bits.  Arrays are (k, j, i) with index -1 at 0."""

    def __init__(self, c, setup):
        w = setup.workload
        self.c, self.work = c, w
        self.im, self.jm, self.km = w.im, w.jm, w.km
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        m = setup.metrics

        def axis(a, lo, n, dim):  # metric with slot x+1 for index x, broadcast along its axis
            full = torch.zeros(n + 4, dtype=torch.float64)
            full[lo + 1: lo + 1 + len(a)] = torch.from_numpy(np.asarray(a, np.float64))
            shape = [1, 1, 1]
            shape[dim] = n + 4
            return full.reshape(shape).to(self.dev)

        self.dx, self.dxs = axis(m["dx1"], -1, w.im, 2), axis(m["dxs"], 0, w.im, 2)
        self.dy, self.dys = axis(m["dy1"], 0, w.jm, 1), axis(m["dys"], 0, w.jm, 1)
        self.dz, self.dzs = axis(m["dzn"], -1, w.km, 0), axis(m["dzs"], -1, w.km, 0)
        k = setup.coeffs
        self.cn = {n: axis(k[n], 1, getattr(w, x), d) for n, x, d in
                   (("cn2l", "im", 2), ("cn2s", "im", 2), ("cn3l", "jm", 1), ("cn3s", "jm", 1), ("cn4l", "km", 0),
                    ("cn4s", "km", 0))}
        ax, by, cz = (torch.from_numpy(np.asarray(t, np.float64)).to(self.dev) for t in k["_cn1_terms"])
        self.cn1 = 1.0 / (ax[None, None, :] + by[None, :, None] + cz[:, None, None])
        top = np.array([m["z2"][q] + np.float32(0.5) * m["dzn"][q + 1] for q in range(1, w.km + 1)], np.float32)
        z = torch.from_numpy(np.ascontiguousarray(setup.zbm.T)).to(self.dev)
        self.mask = (z[None] > torch.from_numpy(top).to(self.dev)[:, None, None]).double()
        self.uin = None if setup.inflow is None else self._plane(setup.inflow)
        z3 = lambda: torch.zeros((w.km + 4, w.jm + 4, w.im + 4), dtype=torch.float64, device=self.dev)  # noqa: E731
        for n in ("u", "v", "w", "p", "f", "g", "h", "fo", "go", "ho", "us", "vs", "ws", "sm"):
            setattr(self, n, z3())
        self.diu = [None] + [z3() for _ in range(9)]
        kk, jj, ii = torch.meshgrid(torch.arange(1, w.km + 1), torch.arange(1, w.jm + 1), torch.arange(1, w.im + 1),
                                    indexing="ij")
        self.red = (((ii + jj + kk) % 2) == 1).to(self.dev)
        self.ro, self.vn, self.dt = float(np.float32(1.1763)), float(setup_gen.VN), float(np.float32(w.dt))
        self.ave = None

    def _plane(self, a):
        return torch.from_numpy(np.ascontiguousarray(np.asarray(a, np.float64).T)).to(self.dev)  # (k, j)

    def s(self, a, di=0, dj=0, dk=0):
        """a on the interior shifted by (di, dj, dk); 1-D metrics along their axis."""
        r = []
        for x, (n, d) in enumerate(((self.km, dk), (self.jm, dj), (self.im, di))):
            r.append(slice(None) if a.shape[x] == 1 else slice(2 + d, 2 + d + n))
        return a[tuple(r)]

    def step(self, n, planes):
        self._velnw()
        self._bondv1(n, planes)
        self._velfg()
        self._les()
        for a, o in (("f", "fo"), ("g", "go"), ("h", "ho")):
            x, y = self.s(getattr(self, a)), self.s(getattr(self, o))
            new = x.clone()
            x.copy_(1.5 * x - 0.5 * y)
            y.copy_(new)
        self._press()

    def _velnw(self):
        s, p = self.s, self.p
        s(self.u).add_(self.dt * (s(self.f) - (s(p, 1) - s(p)) / self.ro / s(self.dxs)))
        s(self.v).add_(self.dt * (s(self.g) - (s(p, 0, 1) - s(p)) / self.ro / s(self.dys)))
        dw = self.dt * (s(self.h) - (s(p, 0, 0, 1) - s(p)) / self.ro / s(self.dzs))
        s(self.w)[:-1].add_(dw[:-1])

    def _bondv1(self, n, planes):
        im, jm, km = self.im, self.jm, self.km
        u, v, w = self.u, self.v, self.w
        K, J = slice(2, km + 2), slice(2, jm + 2)
        if planes is None:
            ins = (self.uin if self.uin is not None else torch.tensor(5.0, dtype=torch.float64), 0.0, 0.0)
        else:
            ins = tuple(self._plane(q) for q in planes)
        hi = im + 1 if n == 1 else 2
        for a, x in zip((u, v, w), ins):
            a[K, J, 1:hi + 1] = x[..., None] if torch.is_tensor(x) and x.dim() == 2 else x
        face = u[K, J, im + 1]
        uout = (torch.clamp(face.max(), min=0.0) + torch.clamp(face.min(), max=0.0)) / 2
        q = self.dt * uout
        u[K, J, im + 1] -= q * (u[K, J, im + 1] - u[K, J, im]) / self.dxs[0, 0, im + 1]
        for a in (v, w):
            a[K, J, im + 2] -= q * (a[K, J, im + 2] - a[K, J, im + 1]) / self.dxs[0, 0, im + 1]
        I = slice(1, im + 3)
        for a, ke in ((u, km + 3), (v, km + 3), (w, km + 2)):
            a[1:ke, 1, I] = a[1:ke, jm + 1, I]
            a[1:ke, jm + 2, I] = a[1:ke, 2, I]
        JJ = slice(1, jm + 3)
        for a in (u, v):
            a[1, JJ, I] = -a[2, JJ, I]
            a[km + 2, JJ, I] = a[km + 1, JJ, I]
        w[1, 0:jm + 3, I] = 0.0
        w[km + 1, 0:jm + 3, I] = 0.0

    def _velfg(self):
        s, u, v, w = self.s, self.u, self.v, self.w
        im, jm, km = self.im, self.jm, self.km
        dx, dy, dz, dzs = self.dx, self.dy, self.dz, self.dzs
        dxi, dxp, dxm = s(dx), s(dx, 1), s(dx, -1)
        dyj, dyp, dym = s(dy), s(dy, 0, 1), s(dy, 0, -1)
        dzk, dzp = s(dz), s(dz, 0, 0, 1)
        z3 = lambda: torch.zeros_like(u)  # noqa: E731
        cov = [None] + [z3() for _ in range(9)]
        D = self.diu

        def put(q, nou, diu, dk=0, keep=None):
            a, b = s(D[q], 0, 0, dk), s(cov[q], 0, 0, dk)
            if keep is not None:
                a[keep], b[keep] = diu[keep], (nou * diu)[keep]
            else:
                a.copy_(diu)
                b.copy_(nou * diu)

        t = (0.5 * (s(v, 0, -1) + s(v))[:1] * dxp + 0.5 * (s(v, 1, -1) + s(v, 1))[:1] * dxi) / (dxi + dxp)
        usp = torch.sqrt(s(u)[:1] ** 2 + t * t)
        t = (0.5 * (s(u, -1) + s(u))[:1] * dyp + 0.5 * (s(u, -1, 1) + s(u, 0, 1))[:1] * dyj) / (dyj + dyp)
        vsp = torch.sqrt(s(v)[:1] ** 2 + t * t)
        put(1, (s(u, -1) + s(u)) / 2, (s(u) - s(u, -1)) / dxi)
        put(5, (s(v, 0, -1) + s(v)) / 2, (s(v) - s(v, 0, -1)) / dyj)
        put(9, (s(w, 0, 0, -1) + s(w)) / 2, (s(w) - s(w, 0, 0, -1)) / dzk)
        put(2, (dxp * s(v, 0, -1) + dxi * s(v, 1, -1)) / (dxi + dxp), 2 * (s(u) - s(u, 0, -1)) / (dym + dyj))
        put(3, (dxp * s(w) + dxi * s(w, 1)) / (dxi + dxp), (s(u, 0, 0, 1) - s(u)) / s(dzs), dk=1)
        put(4, (dyp * s(u, -1) + dyj * s(u, -1, 1)) / (dyj + dyp), 2 * (s(v) - s(v, -1)) / (dxm + dxi))
        put(6, (dyp * s(w) + dyj * s(w, 0, 1)) / (dyj + dyp), (s(v, 0, 0, 1) - s(v)) / s(dzs), dk=1)
        dz1 = float(dz[2, 0, 0])
        wl = math.log(0.5 * dz1 / 0.1)
        for q, vel, sp, nou in ((3, u, usp, 0.5 * (dxp * s(w)[:1] + dxi * s(w, 1)[:1]) / (dxi + dxp)),
                                (6, v, vsp, 0.5 * (dyp * s(w)[:1] + dyj * s(w, 0, 1)[:1]) / (dyj + dyp))):
            d = sp * 0.4 / wl / (0.5 * dz1) / 0.4 * s(vel)[:1] / sp
            s(D[q])[:1], s(cov[q])[:1] = d, nou * d
        keep = slice(0, km - 1)
        put(7, (dzp * s(u, -1) + dzk * s(u, -1, 0, 1)) / (dzk + dzp), 2 * (s(w) - s(w, -1)) / (dxm + dxi), keep=keep)
        put(8, (dzp * s(v, 0, -1) + dzk * s(v, 0, -1, 1)) / (dzk + dzp), 2 * (s(w) - s(w, 0, -1)) / (dym + dyj),
            keep=keep)
        K, J, I = slice(2, km + 2), slice(2, jm + 2), slice(2, im + 2)
        Kw = slice(2, km + 1)
        for a in (D[1], cov[1], D[4], cov[4]):
            a[K, J, im + 2] = a[K, J, im + 1]
        for a in (D[7], cov[7]):
            a[Kw, J, im + 2] = a[Kw, J, im + 1]
        for a, kr in ((D[2], K), (cov[2], K), (D[5], K), (cov[5], K), (D[8], Kw), (cov[8], Kw)):
            a[kr, 1, I] = a[kr, jm + 1, I]
            a[kr, jm + 2, I] = a[kr, 2, I]
        K1, J1, I1 = slice(2, km + 3), slice(2, jm + 3), slice(2, im + 3)
        for a in (D[2], D[3]):
            a[K1, J1, im + 2] = a[K1, J1, im + 1]
        for a in (D[4], D[6]):
            a[K1, 1, I1] = a[K1, jm + 1, I1]
        self.uspd, self.vspd = s(u)[:1] / usp, s(v)[:1] / vsp
        C = cov
        covc = ((dxp * s(C[1]) + dxi * s(C[1], 1)) / (dxi + dxp) + (s(C[2]) + s(C[2], 0, 1)) / 2
                + (s(C[3]) + s(C[3], 0, 0, 1)) / 2)
        df = (2 * (s(D[1], 1) - s(D[1])) / (dxi + dxp) + (s(D[2], 0, 1) - s(D[2])) / dyj
              + (s(D[3], 0, 0, 1) - s(D[3])) / dzk)
        s(self.f).copy_(-covc + self.vn * df)
        covc = ((s(C[4]) + s(C[4], 1)) / 2 + (dyp * s(C[5]) + dyj * s(C[5], 0, 1)) / (dyj + dyp)
                + (s(C[6]) + s(C[6], 0, 0, 1)) / 2)
        df = ((s(D[4], 1) - s(D[4])) / dxi + 2 * (s(D[5], 0, 1) - s(D[5])) / (dyj + dyp)
              + (s(D[6], 0, 0, 1) - s(D[6])) / dzk)
        s(self.g).copy_(-covc + self.vn * df)
        covc = ((s(C[7]) + s(C[7], 1)) / 2 + (s(C[8]) + s(C[8], 0, 1)) / 2
                + (dzp * s(C[9]) + dzk * s(C[9], 0, 0, 1)) / (dzk + dzp))
        df = ((s(D[7], 1) - s(D[7])) / dxi + (s(D[8], 0, 1) - s(D[8])) / dyj + (s(D[9], 0, 0, 1) - s(D[9])) / s(dzs))
        s(self.h)[:-1].copy_((-covc + self.vn * df)[:-1])
        for f, a, vel in (("f", self.us, u), ("g", self.vs, v), ("h", self.ws, w)):  # immersed boundary
            x = s(a)
            x.copy_((x + s(vel)) * self.mask)
            s(getattr(self, f)).add_(-10.0 * x * self.dt - s(vel) * self.mask)

    def _les(self):
        s, D, sm = self.s, self.diu, self.sm
        im, jm, km = self.im, self.jm, self.km
        dxi, dxp, dxm = s(self.dx), s(self.dx, 1), s(self.dx, -1)
        dyj, dyp, dym = s(self.dy), s(self.dy, 0, 1), s(self.dy, 0, -1)
        dzk, dzp, dzm = s(self.dz), s(self.dz, 0, 0, 1), s(self.dz, 0, 0, -1)
        q = 0.25
        uy = (s(D[2], -1) + s(D[2], -1, 1) + s(D[2]) + s(D[2], 0, 1)) * q
        uz = (s(D[3], -1) + s(D[3], -1, 0, 1) + s(D[3]) + s(D[3], 0, 0, 1)) * q
        vx = (s(D[4]) + s(D[4], 0, -1) + s(D[4], 1) + s(D[4], 1, -1)) * q
        vz = (s(D[6], 0, -1) + s(D[6], 0, -1, 1) + s(D[6]) + s(D[6], 0, 0, 1)) * q
        wx = (s(D[7]) + s(D[7], 0, 0, -1) + s(D[7], 1) + s(D[7], 1, 0, -1)) * q
        wy = (s(D[8]) + s(D[8], 0, 0, -1) + s(D[8], 0, 1) + s(D[8], 0, 1, -1)) * q
        a = 0.1 * (self.dx[0, 0, 1] * self.dy[0, 1, 0] * dzk) ** (1.0 / 3.0)
        s(sm).copy_(a * a * torch.sqrt(2 * (s(D[1]) ** 2 + s(D[5]) ** 2 + s(D[9]) ** 2) + (uy + vx) ** 2
                                       + (wy + vz) ** 2 + (uz + wx) ** 2))
        sm[1:km + 3, 0:jm + 3, 1] = sm[1:km + 3, 0:jm + 3, 2]
        sm[1:km + 3, 0:jm + 3, im + 2] = sm[1:km + 3, 0:jm + 3, im + 1]
        sm[1:km + 3, jm + 2, 1:im + 3] = sm[1:km + 3, jm + 1, 1:im + 3]
        sm[1:km + 3, 1, 1:im + 3] = sm[1:km + 3, 2, 1:im + 3]
        sm[1, 0:jm + 3, 1:im + 3] = -sm[2, 0:jm + 3, 1:im + 3]
        sm[km + 2, 0:jm + 3, 1:im + 3] = sm[km + 1, 0:jm + 3, 1:im + 3]

        def mx(dj=0, dk=0):  # between i and i+1
            return (dxp * s(sm, 0, dj, dk) + dxi * s(sm, 1, dj, dk)) / (dxi + dxp)

        def mxm(dj=0, dk=0):  # between i-1 and i
            return (dxi * s(sm, -1, dj, dk) + dxm * s(sm, 0, dj, dk)) / (dxm + dxi)

        t = 0.4 * self.uspd / math.log(0.5 * float(self.dz[2, 0, 0]) / 0.1)
        wallu = t * t * self.uspd
        t = 0.4 * self.vspd / math.log(0.5 * float(self.dz[2, 0, 0]) / 0.1)
        wallv = t * t * self.vspd
        evy2 = (dyp * mx() + dyj * mx(1)) / (dyj + dyp)
        evy1 = (dyp * mx(-1) + dyj * mx()) / (dyj + dyp)
        evz2 = (dzp * mx() + dzk * mx(0, 1)) / (dzk + dzp)
        evz1 = (dzk * mx(0, -1) + dzm * mx()) / (dzm + dzk)
        x = (s(sm, 1) * 2 * s(D[1], 1) - s(sm) * 2 * s(D[1])) / s(self.dxs)
        y = (evy2 * (s(D[2], 0, 1) + s(D[4], 1)) - evy1 * (s(D[2]) + s(D[4], 1, -1))) / dyj
        z1 = evz1 * (s(D[3]) + s(D[7], 1, 0, -1))
        z1[:1] = wallu
        z = (evz2 * (s(D[3], 0, 0, 1) + s(D[7], 1)) - z1) / dzk
        r = x + y + z
        r[:1] += y[:1] + z[:1]
        s(self.f).add_(r)
        evx2 = evy2
        evx1 = (dyp * mxm() + dyj * mxm(1)) / (dyj + dyp)
        x = (evx2 * (s(D[2], 0, 1) + s(D[4], 1)) - evx1 * (s(D[2], -1, 1) + s(D[4]))) / dxi
        y = (s(sm, 0, 1) * 2 * s(D[5], 0, 1) - s(sm) * 2 * s(D[5])) / s(self.dys)
        z1 = evz1 * (s(D[6]) + s(D[8], 0, 1, -1))
        z1[:1] = wallv
        z = (evz2 * (s(D[6], 0, 0, 1) + s(D[8], 0, 1)) - z1) / dzk
        s(self.g).add_(x + y + z)
        evx2 = evz2
        evx1 = (dzp * mxm() + dzk * mxm(0, 1)) / (dzk + dzp)
        my = lambda dk: (dyp * s(sm, 0, 0, dk) + dyj * s(sm, 0, 1, dk)) / (dyj + dyp)  # noqa: E731
        mym = lambda dk: (dyj * s(sm, 0, -1, dk) + dym * s(sm, 0, 0, dk)) / (dym + dyj)  # noqa: E731
        evy2 = (dzp * my(0) + dzk * my(1)) / (dzk + dzp)
        evy1 = (dzp * mym(0) + dzk * mym(1)) / (dzk + dzp)
        x = (evx2 * (s(D[3], 0, 0, 1) + s(D[7], 1)) - evx1 * (s(D[3], -1, 0, 1) + s(D[7]))) / dxi
        y = (evy2 * (s(D[6], 0, 0, 1) + s(D[8], 0, 1)) - evy1 * (s(D[6], 0, -1, 1) + s(D[8]))) / dyj
        z = (s(sm, 0, 0, 1) * 2 * s(D[9], 0, 0, 1) - s(sm) * 2 * s(D[9])) / dzk
        s(self.h).add_(x + y + z)

    def _press(self):
        s, f, g, h, p = self.s, self.f, self.g, self.h, self.p
        im, jm, km = self.im, self.jm, self.km
        K, J, I = slice(2, km + 2), slice(2, jm + 2), slice(2, im + 2)
        f[K, J, 1] = f[K, J, 2]
        g[K, 1, I] = g[K, jm + 1, I]
        h[1, J, I] = 0.0
        h[km + 1, J, I] = 0.0
        dxi, dyj, dzk = s(self.dx), s(self.dy), s(self.dz)

        def div(a, b, c):
            return (s(a) - s(a, -1)) / dxi + (s(b) - s(b, 0, -1)) / dyj + (s(c) - s(c, 0, 0, -1)) / dzk

        rhs = div(f, g, h) + div(self.u, self.v, self.w) / self.dt
        vol = dxi * dyj * dzk
        rhs -= (vol * rhs).sum() / vol.sum()
        co = {n: s(a) for n, a in self.cn.items()}
        other = ~self.red
        for _ in range(self.work.nmaxp // 4 * 4 if self.c["dc"] else self.work.nmaxp):
            sor = 0.0
            for m in (self.red, other):
                t = co["cn2l"] * s(p, 1)
                t.addcmul_(co["cn2s"], s(p, -1)).addcmul_(co["cn3l"], s(p, 0, 1)).addcmul_(co["cn3s"], s(p, 0, -1))
                t.addcmul_(co["cn4l"], s(p, 0, 0, 1)).addcmul_(co["cn4s"], s(p, 0, 0, -1)).sub_(rhs).mul_(self.cn1)
                t.sub_(s(p)).mul_(m)
                if self.work.omega != 1.0:
                    t.mul_(float(np.float32(self.work.omega)))
                s(p).add_(t)
                sor = sor + (t * t).sum()
                self._bound_ij()
            self._bound_k()
            if not self.c["dc"] and float(sor) < self.work.pjuge:
                break
        s(p).sub_((vol * s(p)).sum() / vol.sum())
        self._bound_ij()
        self._bound_k()

    def _bound_ij(self):
        p, im, jm, km = self.p, self.im, self.jm, self.km
        p[1:km + 3, 1:jm + 3, 1] = p[1:km + 3, 1:jm + 3, 2]
        p[1:km + 3, 1:jm + 3, im + 2] = p[1:km + 3, 1:jm + 3, im + 1]
        p[1:km + 3, 1, 1:im + 3] = p[1:km + 3, jm + 1, 1:im + 3]
        p[1:km + 3, jm + 2, 1:im + 3] = p[1:km + 3, 2, 1:im + 3]

    def _bound_k(self):
        p, im, jm, km = self.p, self.im, self.jm, self.km
        p[1, 1:jm + 3, 1:im + 3] = p[2, 1:jm + 3, 1:im + 3]
        p[km + 2, 1:jm + 3, 1:im + 3] = p[km + 1, 1:jm + 3, 1:im + 3]

    def aveflow(self, n, n1, nmax):
        s, u, v, w = self.s, self.u, self.v, self.w
        names = layout.AVE_FIELDS
        if self.ave is None:
            self.ave = {x: torch.zeros_like(u) for x in names}
        A = self.ave
        K0 = (slice(1, self.km + 2), slice(2, self.jm + 2))
        I, I1 = slice(2, self.im + 2), slice(2, self.im + 3)
        if n >= n1:
            for x, y in (("avev", s(v)), ("avep", s(self.p)), ("aveuu", s(u) ** 2), ("avevv", s(v) ** 2),
                         ("aveww", s(w) ** 2), ("avesm", s(self.sm)), ("avesmsm", s(self.sm) ** 2),
                         ("uwfx", 0.25 * (s(u, 0, 0, -1) + s(u)) * (s(w, 0, 0, -1) + s(w, 1, 0, -1)))):
                s(A[x]).add_(y)
            A["aveu"][K0 + (I,)] += u[K0 + (I,)]
            A["avew"][K0 + (I1,)] += w[K0 + (I1,)]
        if n == nmax:
            for x in names:
                A[x] /= nmax - n1 + 1
            s(A["uwfx"]).sub_(0.25 * (s(A["aveu"], 0, 0, -1) + s(A["aveu"])) *
                              (s(A["avew"], 0, 0, -1) + s(A["avew"], 1, 0, -1)))
            for x, y in (("aveuu", "aveu"), ("avevv", "avev"), ("aveww", "avew")):
                s(A[x]).copy_(torch.sqrt(torch.abs(s(A[x]) - s(A[y]) ** 2)))

    def results(self):
        out = {n: self._out(n, getattr(self, n)) for n in FIELDS}
        if self.ave is not None:
            out.update({n: self._out(n, a) for n, a in self.ave.items()})
        return out

    def _out(self, name, a):
        lb, ext = layout.field_shape(name, self.im, self.jm, self.km)
        r = tuple(slice(lo + 1, lo + 1 + n) for lo, n in zip(lb, ext))
        return a.permute(2, 1, 0)[r]
