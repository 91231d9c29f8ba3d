"""Performance cases: whole simulations through the solver factory and the
batch class, as a user's program runs them.

A case names a scenario recipe of mbsolve_amd.setups, the number of levels,
the numerical form (the suffix of the hip-fdtd-* solver name: "" is the plain
FP64 form, the default of a user who switches from the reference), the grid
and the number of time steps.  One pass is mbh_reset + run() + the result
arrays: the state rewound, every time step, and all records on the host.

Forms whose state or generator product holds no more than about 22 bits
("mixed", "mfma": FP32 state; "mfma64": split FP16 product) hand their
records on as float32; their launch geometry is chosen by timing when the
solver is made, and where the state is rounded depends on it.  The FP64 forms
hand on float64.
"""
import math

import numpy as np
import torch

HBAR = 1.05457266e-34
PI = math.atan(1.0) * 4.0
MU0 = PI * 4e-7
EPS0 = 8.854187817e-12
E0 = 1.60217733e-19

SINGLE = ("mixed", "mfma", "mfma64")


def listed():
    return [
        # the smallest call: song2005 of the reference's tool, one grid
        # point, 10000 steps, four point records at every step (latency of
        # a single wavefront's chain and of the launches)
        {"name": "song_point_fp64", "setup": "song", "levels": 3, "form": "",
         "cells": 1, "steps": 10000},
        # ziolkowski1995 of the reference's tool at its own 32768 cells and
        # 200 fs: two-level Cayley in the plain FP64 form, 81 field and
        # inversion snapshots
        {"name": "ziolkowski_fp64", "setup": "ziolkowski", "levels": 2,
         "form": "", "cells": 32768, "steps": 26200, "rows": 81},
        # the single self-induced-transparency run of the benchmark, full
        # length, with its 256 snapshots, FP64-state Bloch form
        {"name": "sit2_zform", "setup": "sit", "levels": 2, "form": "zform",
         "cells": 8192, "steps": 49114, "rows": 256},
        # a batched two-level sweep (the default benchmark workload with
        # fewer runs and a fifth of the steps, same snapshots per step),
        # FP32-state Bloch form, uneven grids of 2^12..2^17 cells
        {"name": "sweep2_mixed", "setup": "sit_sweep", "levels": 2,
         "form": "mixed", "runs": 24, "min_cells": 4096,
         "max_cells": 131072, "steps": 9824, "rows": 4},
        # colliding-pulse mode locking of the reference's tool: gain /
        # absorber / gain, lossy, two density materials: the general
        # two-level Bloch kernel
        {"name": "cpml_zform", "setup": "cpml", "levels": 2, "form": "zform",
         "cells": 8192, "steps": 20000, "rows": 17},
        # the three-level V workload of the benchmark on the matrix cores
        {"name": "v3_mfma64", "setup": "v3", "levels": 3, "form": "mfma64",
         "cells": 65536, "steps": 20000, "rows": 16},
        # the same device in the plain FP64 Rodrigues form
        {"name": "v3_fp64", "setup": "v3", "levels": 3, "form": "",
         "cells": 16384, "steps": 8000, "rows": 16},
        # six-level quantum-cascade gain medium on the matrix cores
        {"name": "qcl6_mfma64", "setup": "qcl", "levels": 6,
         "form": "mfma64", "cells": 262144, "steps": 2000, "rows": 4},
        # six-level bias sweep in the FP64 rotated-basis form (the form of
        # full-length six-level runs), uneven grids
        {"name": "sweep6_zform", "setup": "qcl_sweep", "levels": 6,
         "form": "zform", "runs": 8, "min_cells": 8192, "max_cells": 65536,
         "steps": 1000, "rows": 4},
        # marskar2011 of the reference's tool (six-level ladder, strong
        # pulse) at its own 8192 cells in the plain FP64 form, the first
        # steps, the pulse shortened with them
        {"name": "marskar6_fp64", "setup": "ladder", "levels": 6, "form": "",
         "cells": 8192, "steps": 800, "rows": 16},
        # tzenov2016 of the reference's tool (five-level comb laser starting
        # from noise, which needs the plain FP64 form), the first steps
        {"name": "tzenov5_fp64", "setup": "comb", "levels": 5, "form": "",
         "cells": 8192, "steps": 600, "rows": 4},
        # pure Maxwell line, FP32 state, a long grid with point records
        {"name": "line_mixed", "setup": "line", "levels": 0, "form": "mixed",
         "cells": 1 << 22, "steps": 4000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _steps(rng, lo, hi, cells, budget):
    """Steps log-uniform in [lo, hi] with cells * steps within the budget."""
    hi = max(lo, min(hi, int(budget / cells)))
    return _log_int(rng, lo, hi)


def draw(rng):
    """One more case: a random setup, form, grid and length."""
    setup = rng.choice(["sit", "sit_sweep", "cpml", "v3", "v3_cayley",
                        "ladder", "qcl", "qcl_sweep", "comb", "line"])
    c = {"setup": setup, "levels": 2, "rows": rng.randint(3, 24)}
    if setup == "sit":
        c["form"] = rng.choice(["", "zform", "mixed"])
        c["cells"] = _log_int(rng, 600, 40000)
        c["steps"] = _steps(rng, 4000, 30000, c["cells"], 5e8)
    elif setup == "sit_sweep":
        c["form"] = rng.choice(["", "zform", "mixed"])
        c["runs"] = rng.randint(3, 24)
        c["min_cells"] = _log_int(rng, 1000, 8000)
        c["max_cells"] = _log_int(rng, 10000, 131072)
        c["rows"] = rng.randint(2, 4)
        mean = 0.5 * (c["min_cells"] + c["max_cells"])
        c["steps"] = _steps(rng, 1000, 9824, c["runs"] * mean,
                            1.2e9 if c["form"] == "" else 8e9)
    elif setup == "cpml":
        c["form"] = rng.choice(["", "zform", "mixed"])
        c["cells"] = _log_int(rng, 1000, 16384)
        c["steps"] = _steps(rng, 4000, 20000, c["cells"], 1.6e8)
    elif setup == "v3":
        c["levels"] = 3
        c["form"] = rng.choice(["", "zform", "mixed", "mfma", "mfma64"])
        c["cells"] = _log_int(rng, 2000, 65536)
        c["steps"] = _steps(rng, 1000, 20000, c["cells"],
                            1.3e8 if c["form"] == "" else 1.3e9)
    elif setup == "v3_cayley":
        c["levels"] = 3
        c["form"] = ""
        c["cells"] = _log_int(rng, 1000, 16384)
        c["steps"] = _steps(rng, 500, 8000, c["cells"], 3e7)
    elif setup == "ladder":
        c["levels"] = rng.randint(4, 6)
        c["form"] = rng.choice(["", "zform", "mixed", "mfma", "mfma64"])
        if c["form"] == "":
            c["cells"] = _log_int(rng, 300, 8192)
            c["steps"] = _log_int(rng, 300, 800)
        else:
            c["cells"] = _log_int(rng, 2000, 65536)
            c["steps"] = _steps(rng, 800, 8000, c["cells"], 1.5e8)
    elif setup == "qcl":
        c["levels"] = 6
        c["form"] = rng.choice(["zform", "mfma", "mfma64"])
        c["cells"] = _log_int(rng, 4096, 262144)
        c["steps"] = _steps(rng, 500, 4000, c["cells"], 4e8)
        c["rows"] = rng.randint(2, 4)
    elif setup == "qcl_sweep":
        c["levels"] = 6
        c["form"] = rng.choice(["zform", "mfma", "mfma64"])
        c["runs"] = rng.randint(2, 8)
        c["min_cells"] = _log_int(rng, 2000, 8000)
        c["max_cells"] = _log_int(rng, 10000, 65536)
        c["rows"] = rng.randint(2, 4)
        mean = 0.5 * (c["min_cells"] + c["max_cells"])
        c["steps"] = _steps(rng, 300, 2000, c["runs"] * mean, 2e8)
    elif setup == "comb":
        c["levels"] = 5
        c["form"] = ""
        c["cells"] = _log_int(rng, 1000, 8192)
        c["steps"] = _steps(rng, 300, 1500, c["cells"], 4e6)
        c["rows"] = rng.randint(2, 8)
    else:
        c["levels"] = 0
        c["form"] = rng.choice(["", "mixed"])
        c["cells"] = _log_int(rng, 4096, 1 << 22)
        c["steps"] = _steps(rng, 2000, 8000, c["cells"], 1.6e10)
        c["rows"] = 0
    return c


# ------------------------------------------------------------- scenarios ---
def _end(length, cells, steps, eps_min):
    """End time for which the grid rule gives `steps` time steps."""
    dt = 0.5 * length / (cells - 1) * math.sqrt(MU0 * EPS0 * eps_min)
    return (steps - 1.5) * dt


def _sech(spec, areas, dipoles):
    """Sech pulses of the given areas, their peak inside the run: a run of
    1.5 ps has the recipe's 1 / beta = 100 fs."""
    from mbsolve_amd import setups
    beta = 15.0 / spec["endtime"]
    for s, area, d in zip(spec["sources"], areas, dipoles):
        s["beta"], s["phase"] = beta, 7.0
        s["ampl"] = setups.sech_area_amplitude(area, beta, d)


def _snapshots(spec, rows):
    spec["records"] = [r for r in spec["records"]
                       if "type" in r or r.get("position", -1.0) >= 0.0]
    if rows:
        iv = spec["endtime"] / (rows - 1)
        spec["records"] += [{"name": "inv12", "interval": iv},
                            {"name": "e", "interval": iv}]


def _specs(case, seed):
    """The scenario recipes of a case with the seed's pulse areas, rates,
    amplitudes and initial values."""
    from mbsolve_amd import setups
    rng = np.random.default_rng(seed)
    kind, steps, rows = case["setup"], case["steps"], case.get("rows", 0)
    cells = case.get("cells", 0)

    def sit(n, length, name):
        s = setups.sit_2lvl(
            num_gridpoints=n, length=length, name=name,
            endtime=_end(length, n, steps, 1.0),
            t2=10 ** rng.uniform(math.log10(10e-15), math.log10(1e-9)))
        _sech(s, [rng.uniform(0.5 * PI, 4 * PI)], [1e-29])
        _snapshots(s, rows)
        return s

    def uneven():
        # the grids belong to the case, the devices on them to the seed
        grid = np.random.default_rng(case["runs"])
        return [int(round(math.exp(u)))
                for u in grid.uniform(math.log(case["min_cells"]),
                                      math.log(case["max_cells"]),
                                      size=case["runs"])]

    if kind == "sit":
        return [sit(cells, 150e-6, "sit2")]
    if kind == "sit_sweep":
        dx = 150e-6 / 8191
        return [sit(n, dx * (n - 1), "s%02d" % r)
                for r, n in enumerate(uneven())]
    if kind == "qcl_sweep":
        out = []
        for r, n in enumerate(uneven()):
            bias = 0.9 + 0.2 * r / max(1, case["runs"] - 1)
            out.append(setups.qcl6(
                num_gridpoints=n, num_timesteps=steps, bias=bias,
                seed=int(rng.integers(1 << 30)), num_records=rows,
                name="q%02d" % r))
        return out
    if kind == "qcl":
        return [setups.qcl6(num_gridpoints=cells, num_timesteps=steps,
                            seed=int(rng.integers(1 << 30)),
                            num_records=rows)]
    if kind == "song":
        s = setups.song2005(num_timesteps=steps)
        s["sources"][0]["ampl"] *= rng.uniform(0.5, 1.0)
    elif kind == "ziolkowski":
        s = setups.ziolkowski1995(num_gridpoints=cells)
        s["endtime"] = _end(150e-6, cells, steps, 1.0)
        s["sources"][0]["ampl"] *= rng.uniform(0.5, 1.0)
        _snapshots(s, rows)
    elif kind == "cpml":
        s = setups.tzenov2018_cpml(num_gridpoints=cells)
        s["endtime"] = _end(1.125e-3, cells, steps, 12.96)
        s["rho_init"] = ([0.5, 0.5], [1e-3 * rng.uniform(0.5, 1.5)])
        _snapshots(s, rows)
    elif kind in ("v3", "v3_cayley"):
        s = setups.v3_rodr(num_gridpoints=cells,
                           endtime=_end(150e-6, cells, steps, 1.0),
                           algo="cvr-rodr" if kind == "v3" else "reg-cayley")
        _sech(s, rng.uniform(0.5 * PI, 3 * PI, size=2), [1e-29, 0.8e-29])
        _snapshots(s, rows)
    elif kind == "ladder":
        length = 1e-3 / 8191 * (cells - 1)
        s = setups.marskar2011(num_levels=case["levels"],
                               num_gridpoints=cells,
                               endtime=_end(length, cells, steps, 1.0))
        s["regions"] = [("Active region", "AR_Marsk", 0.0, length)]
        tau = min(100e-15, s["endtime"] / 6.0)
        s["sources"][0].update(tau=tau, phase=3.0 * tau,
                               ampl=5e8 * rng.uniform(0.5, 1.0))
        _snapshots(s, rows)
    elif kind == "comb":
        s = setups.tzenov2016(num_gridpoints=cells,
                              seed=int(rng.integers(1 << 30)),
                              endtime=_end(5e-3, cells, steps, 19.35))
        a = rng.uniform(0.0, 0.2)
        s["rho_init"] = ([a, 0.0, 1.0 - a, 0.0, 0.0], [])
        _snapshots(s, rows)
    elif kind == "line":
        s = setups.maxwell_line(num_gridpoints=cells, num_timesteps=steps)
        s["sources"][0]["ampl"] *= rng.uniform(0.5, 1.0)
        s["records"] += [
            {"name": "e1", "interval": 0.0, "position": 90e-9},
            {"name": "h1", "interval": 0.0, "position": 700e-9}]
    else:
        raise ValueError(kind)
    return [s]


# --------------------------------------------------------- prepare / run ---
def prepare(case, seed):
    import mbsolve_amd.lib as mb
    import mbsolve_amd.solverhip  # noqa: F401
    from mbsolve_amd import setups
    specs = _specs(case, seed)
    name = setups.solver_name(specs[0], case["form"])
    if "runs" in case:
        mb.material.clear_library()
        sol = mb.solver_hip_batch(
            name, [setups.build(s, clear_library=False) for s in specs])
        results = [sol.get_results(r) for r in range(len(specs))]
    else:
        dev, scen = setups.build(specs[0])
        sol = mb.solver.create_instance(name, dev, scen)
        results = [sol.get_results()]
    return {"solver": sol, "results": results,
            "single": case["form"] in SINGLE}


def run(state):
    state["solver"].reset()
    state["solver"].run()
    out = []
    for results in state["results"]:
        got = [r.get_data_real() for r in results]
        if state["single"]:
            got = [x.astype(np.float32) for x in got]
        out.append(got)
    return out


def work(case):
    """The state and the sources read once, the state and the records written
    once; per cell and step the Yee update and, with N levels, a dense
    (N^2 - 1)^2 propagator step with its rotation and polarization."""
    n, steps = case["levels"], case["steps"]
    if "runs" in case:
        a, b = case["min_cells"], case["max_cells"]
        cells = case["runs"] * (b - a) / math.log(b / a)
    else:
        cells = case["cells"]
    k = n * n - 1 if n else 0
    size = 4 if case["form"] in ("mixed", "mfma") else 8
    rec = 2 * case.get("rows", 0) * cells
    rec += steps * {"song": 4, "ladder": n + 1, "comb": 6, "cpml": 2,
                    "line": 3}.get(case["setup"], 0)
    nbytes = 2 * cells * size * (2 + (1 + k if n else 0)) + 8 * (rec + steps)
    flops = cells * steps * (10 + (2 * k * k + 5 * k if n else 0))
    return {"bytes": float(nbytes), "flops": float(flops)}


# ----------------------------------------------------------------- exact ---
def exact(case, seed):
    """The same simulations in plain torch, FP64 / complex128: Yee leapfrog
    and, per cell, the Cayley step of the 2 x 2 density matrix as a rotation
    of its Bloch vector, or the Strang step of the Lindblad equation
    (dipole rotation between two exponential half steps) of the N x N density
    matrix in the eigenbasis of the dipole operator."""
    if case["setup"] == "v3_cayley":
        return None  # a matrix inverse per cell and step: too slow in torch
    specs = _specs(case, seed)
    cells = sum(s["num_gridpoints"] for s in specs)
    n = case["levels"]
    per_step = 2.5e-4 + cells * (4e-10 if n < 3 else 2.5e-10 * n * n)
    per_step += 1.2e-4 * (len(specs) if n > 2 else 0)
    if case["steps"] * per_step > 18.0:
        return None
    out = _Exact(specs, n).run()
    if case["setup"] == "comb":
        # E starts from 1e-15 V/m: below the rounding of p in this basis
        out = [[None if s["name"][0] == "e" else r
                for s, r in zip(specs[0]["records"], out[0])]]
    return out


def _matrix(diag, off, n):
    m = np.zeros((n, n), dtype=complex)
    m[np.arange(n), np.arange(n)] = diag
    it = iter(off)
    for col in range(n):
        for row in range(col):
            v = complex(next(it, 0.0))
            m[row, col], m[col, row] = v, v.conjugate()
    return m


def _expm(A):
    """Taylor series of exp(A / 2^k) - I, then squared k times in the form
    (I + X)^2 - I (no cancellation against the identity)."""
    k = max(0, int(math.ceil(math.log2(max(np.abs(A).sum(axis=1).max(),
                                           1e-300)))) + 4)
    A = A / 2.0 ** k
    X = np.zeros_like(A)
    for j in range(14, 0, -1):
        X = (A + A @ X) / j
    for _ in range(k):
        X = 2.0 * X + X @ X
    return np.eye(len(A)) + X


class _Medium:
    """H0, mu, population rates s and coherence rates d of a medium."""

    def __init__(self, q):
        if q.get("type") == "2lvl":
            g, w = q["scattering_rate"], q.get("equilibrium_inversion", -1.0)
            f = HBAR * q["transition_freq"] / 2
            q = {"num_levels": 2, "carrier_density": q["carrier_density"],
                 "h_diag": [-f, f], "h_off": [0.0], "mu_diag": [0.0, 0.0],
                 "mu_off": [-E0 * q["dipole_moment"]],
                 "scattering": [[0.0, g * 0.5 * (1 - w)],
                                [g * 0.5 * (1 + w), 0.0]],
                 "pure_dephasing": [q["dephasing_rate"] - 0.5 * g]}
        n = self.n = q["num_levels"]
        self.density = q["carrier_density"]
        self.H = _matrix(q["h_diag"], q["h_off"], n)
        self.mu = _matrix(q["mu_diag"], q["mu_off"], n)
        s = np.array(q["scattering"], dtype=float)
        s[np.arange(n), np.arange(n)] = 0.0
        s[np.arange(n), np.arange(n)] = -s.sum(axis=0)
        self.s = s
        self.d = np.zeros((n, n))
        pure = iter(q["pure_dephasing"])
        for col in range(n):
            for row in range(col):
                r = -abs(next(pure)) + 0.5 * (s[row, row] + s[col, col])
                self.d[row, col] = self.d[col, row] = r

    def generator(self):
        """L0 on the row-major vec of rho: -i/hbar [H, .] + D."""
        n = self.n
        eye = np.eye(n)
        L = -1j / HBAR * (np.kron(self.H, eye) - np.kron(eye, self.H.T))
        L = L + np.diag(self.d.ravel()).astype(complex)
        for i in range(n):
            for j in range(n):
                L[i * n + i, j * n + j] += self.s[i, j]
        return L


class _Exact:
    def __init__(self, specs, n):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.n, self.specs = n, specs
        self.runs, base = [], 0
        fa, fb, fc, fg, fx, e0, med = [], [], [], [], [], [], []
        for s in specs:
            r = self._grid(s)
            r["base"] = base
            nx = r["nx"]
            idx = np.full(nx, -1)
            x = np.arange(nx) * r["dx"]
            names = []
            for k, (_, mid, a, b) in enumerate(s["regions"]):
                names.append(mid)
                idx[(idx < 0) & (x >= a) & (x <= b)] = k
            cols = np.zeros((5, nx))
            for k, mid in enumerate(names):
                m = s["materials"][mid]
                eps = m.get("rel_permittivity", 1.0)
                mur = m.get("rel_permeability", 1.0)
                sig = math.sqrt(EPS0 * eps / (MU0 * mur)) * \
                    m.get("losses", 0.0) * 2.0
                y = sig * r["dt"] / (2.0 * EPS0 * eps)
                w = idx == k
                cols[0, w] = (1.0 - y) / (1.0 + y)
                cols[1, w] = r["dt"] / (EPS0 * eps) / (1.0 + y)
                cols[2, w] = r["dt"] / (MU0 * mur * r["dx"])
                cols[3, w] = m.get("overlap_factor", 1.0)
                cols[4, w] = 1.0 / r["dx"]
                if m.get("qm"):
                    at = np.nonzero(w)[0]
                    if at.size:
                        med.append((base + at[0], base + at[-1] + 1,
                                    _Medium(m["qm"]), s["rho_init"],
                                    r["dt"]))
            # one cell between runs holds the boundary H of the run before
            pad = np.zeros(1)
            for lst, c in zip((fa, fb, fc, fg, fx), cols):
                lst += [c, pad]
            e0 += [np.full(nx, s.get("e_init", 0.0)), pad]
            self.runs.append(r)
            base += nx + 1
        self.G = base
        t = self._t
        self.fa = t(np.concatenate(fa))
        fbv = np.concatenate(fb)
        self.fp = t(-fbv * np.concatenate(fg))
        self.fh = t(fbv * np.concatenate(fx))
        fcv = np.concatenate(fc)
        for r in self.runs:
            fcv[r["base"]] = 0.0
        self.fc = t(fcv)
        self.e = t(np.concatenate(e0))
        self.h = torch.zeros_like(self.e)
        self.p = torch.zeros_like(self.e)
        self.algo = specs[0]["algo"]
        if self.algo == "reg-cayley":
            self._cayley(med)
        elif self.algo == "cvr-rodr":
            self._rodr(med)

    def _t(self, a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(self.dev)

    @staticmethod
    def _grid(s):
        nx = s["num_gridpoints"]
        length = sum(b - a for _, _, a, b in s["regions"])
        eps = min(s["materials"][m].get("rel_permittivity", 1.0)
                  for _, m, _, _ in s["regions"])
        if nx == 1:
            dx, nt = 1e13, s["num_timesteps"]
        else:
            dx = length / (nx - 1)
            nt = int(math.ceil(s["endtime"] /
                               (0.5 * dx * math.sqrt(MU0 * EPS0 * eps))) + 1)
        dt = s["endtime"] / (nt - 1)
        tt = np.arange(nt) * dt
        src = []
        for q in s.get("sources", []):
            if q["kind"] == "sech":
                v = np.sin(2 * PI * q["freq"] * tt - q.get("phase_sin", 0.0))
                v = v / np.cosh(q["beta"] * tt - q["phase"])
            elif q["kind"] == "gauss":
                v = np.exp(-(tt - q["phase"]) ** 2 / q["tau"] ** 2)
                v = v * np.sin(2 * PI * q["freq"] * tt)
            else:
                v = np.sin(2 * PI * q["freq"] * tt + q.get("phase", 0.0))
            src.append((int(q["position"] / dx), q.get("hard", True),
                        q["ampl"] * v))
        recs = []
        for q in s["records"]:
            iv = q.get("interval", 0.0)
            rows = nt if iv <= dt else int(math.floor(s["endtime"] / iv)) + 1
            ratio = 1.0 if iv <= dt else dt / iv
            pos = q.get("position", -1.0)
            at = None if pos < 0.0 else int(round(pos / dx))
            kind = {"e": 0, "p": 1, "h": 2, "d": 3, "i": 4}[q["name"][0]]
            recs.append({"kind": q.get("type", kind), "row": q.get("row", 1),
                         "rows": rows, "ratio": ratio, "at": at})
        return {"nx": nx, "dx": dx, "nt": nt, "dt": dt, "src": src,
                "recs": recs}

    # ---- two-level Cayley, constants per cell ----------------------------
    def _cayley(self, med):
        G = self.G
        z = {k: np.zeros(G) for k in
             ("bz", "be", "A0", "g", "D00", "D01", "D10", "D11", "px", "py",
              "r0", "r1", "mx", "my")}
        z["A0"][:] = 1.0
        for a, b, m, (diag, off), dt in med:
            k = dt / HBAR
            z["bz"][a:b] = k * (m.H[0, 0] - m.H[1, 1]).real / 2
            z["be"][a:b] = -k * m.mu[0, 1].real
            z["A0"][a:b] = 1.0 + (k * (m.H[0, 0] + m.H[1, 1]).real / 4) ** 2
            z["g"][a:b] = math.exp(m.d[0, 1] * dt / 2)
            D = _expm(m.s * dt / 2)
            z["D00"][a:b], z["D01"][a:b] = D[0]
            z["D10"][a:b], z["D11"][a:b] = D[1]
            # p = n tr(mu d rho/dt) at zero field, linear in rho01
            w = (m.H[0, 0] - m.H[1, 1]).real / HBAR
            mu = m.mu[0, 1].real
            z["px"][a:b] = 2 * m.density * mu * m.d[0, 1]
            z["py"][a:b] = 2 * m.density * mu * w
            rho = _matrix(diag, off, 2)
            z["r0"][a:b], z["r1"][a:b] = rho[0, 0].real, rho[1, 1].real
            z["mx"][a:b], z["my"][a:b] = rho[0, 1].real, -rho[0, 1].imag
        for k, v in z.items():
            setattr(self, k, self._t(v))
        self.bz2 = self.bz * self.bz
        self._dissipate()  # the first half step of step 0

    def _dissipate(self):
        self.mx *= self.g
        self.my *= self.g
        r0 = self.D00 * self.r0 + self.D01 * self.r1
        self.r1 = self.D10 * self.r0 + self.D11 * self.r1
        self.r0 = r0

    def _step_cayley(self):
        bx = self.be * self.e
        r2 = torch.addcmul(self.bz2, bx, bx)
        sc = torch.sub(self.A0, r2, alpha=0.25)
        lam = 2.0 / torch.addcmul(r2, sc, sc)
        mz = 0.5 * (self.r0 - self.r1)
        c = self.bz * self.mx - bx * mz
        w, g = lam * self.my, lam * c
        q = torch.addcmul(g, sc, w)
        self.mx = torch.addcmul(self.mx, self.bz, q, value=-1.0)
        up = bx * q
        self.r0 += up
        self.r1 -= up
        self.my = self.my + sc * g - r2 * w
        self._dissipate()  # second half step: the state of this step
        # rho01 = mx - i my:  d rho01/dt = (-i w + d) rho01
        self.p = torch.addcmul(self.px * self.mx, self.py, self.my,
                               value=-1.0)
        self.after = True

    # ---- Rodrigues: vec(rho) in the dipole eigenbasis, medium by medium --
    def _rodr(self, med):
        n, self.media = self.n, []
        for a, b, m, (diag, off), dt in med:
            lam, S = np.linalg.eigh(m.mu)
            T = np.kron(S.conj().T, S.T)
            L = m.generator()
            E = _expm(L * dt / 2)
            Tinv = T.conj().T
            rho = _matrix(diag, off, n).ravel()
            back = E @ Tinv
            y = (T @ (E @ rho))[:, None] * np.ones((1, b - a))
            pv = m.density * (m.mu.T.ravel() @ L @ back)
            self.media.append({
                "a": a, "b": b, "y": self._t(y),
                "ph": self._t(lam * dt / HBAR)[:, None],
                "W": self._t(T @ E @ E @ Tinv), "p": self._t(pv),
                "pop": self._t(back[np.arange(n) * (n + 1)])})

    def _step_rodr(self):
        for m in self.media:
            a, b, n = m["a"], m["b"], self.n
            ang = m["ph"] * self.e[a:b]
            u = torch.complex(torch.cos(ang), torch.sin(ang))
            y = m["y"].view(n, n, b - a)
            y = y * u[:, None, :] * u.conj()[None, :, :]
            m["r"] = y.reshape(n * n, b - a)
            self.p[a:b] = (m["p"] @ m["r"]).real
            m["y"] = m["W"] @ m["r"]

    def _population(self, i):
        """rho_ii of all cells (1 / N without a medium: the zero coherence
        vector of the Rodrigues solvers)."""
        if self.algo == "reg-cayley":
            return (self.r0, self.r1)[i]
        out = torch.full_like(self.e, 1.0 / self.n)
        for m in self.media:
            out[m["a"]:m["b"]] = (m["pop"][i] @ m["r"]).real
        return out

    def _step_density(self):
        if self.algo == "cvr-rodr":
            self._step_rodr()
        elif self.algo == "reg-cayley":
            if getattr(self, "after", False):
                self._dissipate()  # the first half step of this step
            self._step_cayley()

    def run(self):
        nt = self.runs[0]["nt"]
        out = [[np.zeros((q["rows"], r["nx"] if q["at"] is None else 1))
                for q in r["recs"]] for r in self.runs]
        # point records stay on the device until the end
        point = [[torch.zeros(q["rows"], dtype=torch.float64,
                              device=self.dev) if q["at"] is not None
                  else None for q in r["recs"]] for r in self.runs]
        src = [(r["base"] + i, hard, self._t(v)) for r in self.runs
               for i, hard, v in r["src"]]
        for n in range(nt):
            e = self.fa * self.e
            if self.algo != "noop":
                e = torch.addcmul(e, self.fp, self.p)
            e[:-1] += self.fh[:-1] * (self.h[1:] - self.h[:-1])
            for i, hard, v in src:
                if hard:
                    e[i] = v[n]
                else:
                    e[i] += v[n]
            self.e = e
            self.h[1:] += self.fc[1:] * (e[1:] - e[:-1])
            self._step_density()
            for k, r in enumerate(self.runs):
                for j, q in enumerate(r["recs"]):
                    row = math.floor(q["ratio"] * n)
                    if n and math.floor(q["ratio"] * (n - 1)) == row:
                        continue
                    if row >= q["rows"]:
                        continue
                    self._record(r, q, row, out[k][j], point[k][j])
        for k, r in enumerate(self.runs):
            for j, q in enumerate(r["recs"]):
                if q["at"] is not None:
                    out[k][j][:, 0] = point[k][j].cpu().numpy()
        return out

    def _record(self, r, q, row, out, point):
        if q["kind"] == 0:
            v = self.e
        elif q["kind"] == 1:
            v = self.p
        elif q["kind"] == 2:
            v = self.h
        elif self.algo == "noop":
            return
        elif q["kind"] == 3:
            v = self._population(q["row"] - 1)
        else:
            v = self._population(1) - self._population(0)
        if q["at"] is None:
            out[row] = v[r["base"]:r["base"] + r["nx"]].cpu().numpy()
        else:
            point[row] = v[r["base"] + q["at"]]
