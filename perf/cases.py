"""Performance cases of the framework: what a user has it do, through its
public entry points, from the smallest calls to the largest.

Six kinds of work:

* ``laminar``: the H8 SIMPLE solver (``H8.run``) from rest at a Reynolds
  number of the seed, for a fixed number of SIMPLE iterations: straight pipe
  or lid-driven cavity, FP64 or FP32 AMG, the solver settings of the bench
  (FGMRES, Jacobi-smoothed V-cycle) or the H8 binary's defaults (PCG,
  Chebyshev-smoothed V-cycle), with or without the mixing-length and SUPG
  terms;
* ``poisson``: an explicit SPD system with its AMG hierarchy
  (``System.solve``): the P1 Laplacian of a Kuhn cube to 1e-8;
* ``komega``: k-omega SST transport steps on a pipe velocity
  (``H8.turb_step``);
* ``sst``: the coupled k-omega SST SIMPLE loop on the pipe (``H8.run``);
* ``wall``: the wall-function k-omega SST path on the helical pipe
  (``H8.run_window``) from its potential start, CF/PMIS AMG-PCG pressure;
* ``gnn``: inference and one gradient of the learned warm start's network
  (``Gnn.forward``, ``Gnn.gradient``).

Sizes are those of the bench and the tests, and odd ones between them.
Meshes are written once per process group into the temporary folder.
"""
from __future__ import annotations

import functools
import math
import os
import shutil
import tempfile
from pathlib import Path

import numpy as np

from nodals_amd import meshgen, p1
from nodals_amd._lib import H8, Gnn, System


# ----------------------------------------------------------------- the cases
def listed():
    return [
        # lid-driven cavity on a coarse grid: every kernel is a few microseconds,
        # so launches and host round trips count (the cavity's pinned pressure path)
        {"name": "cavity_3k_fp64", "kind": "laminar", "mesh": "cavity", "n": 8, "precision": "fp64",
         "solver": "bench", "terms": "none", "its": 60},
        # the bench's pipe and settings: FP32 AMG inside FGMRES
        {"name": "pipe_40k_fp32", "kind": "laminar", "mesh": "pipe", "core": 8, "ring": 5, "slabs": 30,
         "precision": "fp32", "solver": "bench", "terms": "none", "its": 100},
        # the H8 binary's default solver on a mesh of odd section and slab counts
        {"name": "pipe_64k_defaults", "kind": "laminar", "mesh": "pipe", "core": 9, "ring": 5, "slabs": 41,
         "precision": "fp64", "solver": "defaults", "terms": "none", "its": 40},
        # the largest pipe of the bench (768,768 cells), defaults
        {"name": "pipe_769k_defaults", "kind": "laminar", "mesh": "pipe", "core": 16, "ring": 10, "slabs": 143,
         "precision": "fp64", "solver": "defaults", "terms": "none", "its": 20},
        # the optional momentum terms (mixing length and SUPG) on a small odd pipe
        {"name": "pipe_18k_rans", "kind": "laminar", "mesh": "pipe", "core": 6, "ring": 4, "slabs": 23,
         "precision": "fp64", "solver": "defaults", "terms": "rans", "its": 30},
        # the bench's pressure-Poisson system, FP64 hierarchy
        {"name": "poisson_64_fp64", "kind": "poisson", "n": 64, "precision": "fp64", "smoother": "mcgs"},
        # a small system of odd size with the BF16 hierarchy
        {"name": "poisson_23_bf16", "kind": "poisson", "n": 23, "precision": "bf16", "smoother": "mcgs"},
        # turbulence steps on the bench's pipe
        {"name": "komega_40k", "kind": "komega", "core": 8, "ring": 5, "slabs": 30, "steps": 5},
        # the coupled turbulent loop on the bench's pipe
        {"name": "sst_40k_fp32", "kind": "sst", "core": 8, "ring": 5, "slabs": 30, "precision": "fp32", "its": 10},
        # the bench's helix with wall functions, FP64: the most expensive iteration there is
        {"name": "helix_207k_wall_fp64", "kind": "wall", "core": 12, "ring": 9, "slabs": 60, "precision": "fp64",
         "re": 50000.0, "its": 3},
        # a small helix, FP32 AMG
        {"name": "helix_25k_wall_fp32", "kind": "wall", "core": 6, "ring": 4, "slabs": 32, "precision": "fp32",
         "re": 20000.0, "its": 4},
        # forward and backward of the learned warm start on the bench's pipe
        {"name": "gnn_40k", "kind": "gnn", "core": 8, "ring": 5, "slabs": 30},
    ]


# Cube sizes whose Galerkin operators hold an entry that rounds to zero on one
# side of the diagonal only: the coarse colouring can refuse them.
_ONE_SIDED = {20, 24, 25, 26, 28, 29, 39, 40, 42, 43, 48, 50, 52, 54, 55, 56, 57, 58, 59, 60}


def _section(rng, cells, lo=4, hi=16):
    """(core, ring, slabs) of an O-grid pipe of about `cells` tetrahedra."""
    core = max(lo, min(hi, round((cells / 600.0) ** (1.0 / 3.0) * rng.uniform(0.8, 1.2) * 1.9)))
    ring = max(2, round(core * rng.uniform(0.5, 0.75)))
    quads = core * core + 4 * core * ring
    return core, ring, max(5, round(cells / (6.0 * quads)))


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["laminar", "laminar", "laminar", "poisson", "poisson", "komega", "sst", "wall", "gnn"])
    if kind == "laminar":
        cells = _log(rng, 3e3, 1.5e5)
        its = int(max(15, min(100, 8e6 / cells)))
        solver, terms = rng.choice(["bench", "defaults"]), rng.choice(["none", "none", "none", "rans"])
        precision = rng.choice(["fp64", "fp32"])
        if rng.random() < 0.25:
            n = max(7, round((min(cells, 2e5) / 6.0) ** (1.0 / 3.0)))
            return {"kind": kind, "mesh": "cavity", "n": n, "precision": precision, "solver": "bench",
                    "terms": "none", "its": its}
        core, ring, slabs = _section(rng, cells)
        return {"kind": kind, "mesh": "pipe", "core": core, "ring": ring, "slabs": slabs, "precision": precision,
                "solver": solver, "terms": terms, "its": min(its, 40) if terms == "rans" else its}
    if kind == "poisson":
        n, smoother = round(_log(rng, 12, 64)), rng.choice(["mcgs", "jacobi"])
        return {"kind": kind, "n": n, "precision": rng.choice(["fp64", "fp32", "bf16"]),
                "smoother": "jacobi" if n in _ONE_SIDED else smoother}
    if kind == "komega":
        core, ring, slabs = _section(rng, _log(rng, 1e4, 9e4))
        return {"kind": kind, "core": core, "ring": ring, "slabs": slabs, "steps": 5}
    if kind == "sst":
        core, ring, slabs = _section(rng, _log(rng, 1e4, 9e4))
        return {"kind": kind, "core": core, "ring": ring, "slabs": slabs, "precision": rng.choice(["fp64", "fp32"]),
                "its": 10}
    if kind == "wall":
        core = rng.randint(4, 8)
        return {"kind": kind, "core": core, "ring": rng.randint(3, 6), "slabs": rng.randint(30, 56),
                "precision": rng.choice(["fp64", "fp32"]), "re": float(round(_log(rng, 1e4, 5e4))), "its": 3}
    core, ring, slabs = _section(rng, _log(rng, 5e3, 1e5))
    return {"kind": "gnn", "core": core, "ring": ring, "slabs": slabs}


# ----------------------------------------------------------------- meshes
def _mesh(name, write):
    """Folder of a generated mesh, written once (renamed into place whole)."""
    root = Path(tempfile.gettempdir()) / f"nodals_perf_meshes_{os.getuid()}"
    d = root / name
    if not (d / "boundary").exists():
        root.mkdir(parents=True, exist_ok=True)
        tmp = Path(tempfile.mkdtemp(dir=root))
        write(tmp)
        try:
            os.rename(tmp, d)
        except OSError:  # another process was first
            shutil.rmtree(tmp, ignore_errors=True)
    return str(d)


def _pipe(c):
    return _mesh(f"pipe_{c['core']}_{c['ring']}_{c['slabs']}",
                 lambda d: meshgen.write_pipe_case(d, core=c["core"], ring=c["ring"], nslab=c["slabs"]))


def _cells(c):
    if c.get("mesh") == "cavity":
        return 6 * c["n"] ** 3
    return 6 * c["slabs"] * (c["core"] ** 2 + 4 * c["core"] * c["ring"])


# ----------------------------------------------------------------- states
_BENCH = ["--amg-smoother", "jacobi", "--amg-jacobi-omega", "0.7", "--pressure-solver", "fgmres",
          "--pressure-restart", "30", "--alpha-u", "0.5", "--alpha-p", "0.5"]


def _converge(its):
    """A fixed number of SIMPLE iterations: a tolerance that is not met before."""
    return ["--run-mode", "converge", "--max-outer", str(its), "--simple-tol", "1e-13", "--p-max", "400",
            "--verbose", "0"]


def _laminar(c, rng):
    if c["mesh"] == "cavity":
        mesh = _mesh(f"cavity_{c['n']}", lambda d: meshgen.write_cavity_case(d, n=c["n"]))
        args = ["--mesh", mesh, "--lid", "lid", "--wall", "walls", "--re", repr(rng.uniform(60.0, 140.0)),
                "--p-rtol", "0.1"]
    else:
        re = rng.uniform(150.0, 250.0) if c["terms"] == "rans" else rng.uniform(10.0, 45.0)
        args = ["--mesh", _pipe(c), "--re", repr(re), "--p-rtol", "0.5"]
    if c["terms"] == "rans":
        args += ["--mixing-length", "1", "--mixlen-scale", "0.7", "--supg", "1", "--supg-tau-scale", "0.1",
                 "--supg-magic", "4.0"]
    if c["solver"] == "bench":
        args += _BENCH
    h = H8(args + _converge(c["its"]) + ["--amg-precision", c["precision"]])
    return {"h": h, "rest_p": np.zeros(h.info["cells"]), "rest_u": np.zeros(h.info["nv"])}


def _turb_start(h, s):
    for name, v in (("k", h.turb["k_in"]), ("omega", h.turb["omega_in"])):
        s[name] = np.zeros(h.turb["ns"])
        s[name][:h.turb["nvert"]] = v


def _wall(c, rng):
    mesh = _mesh(f"helix_{c['core']}_{c['ring']}_{c['slabs']}",
                 lambda d: meshgen.write_helix_case(d, core=c["core"], ring=c["ring"], nslab=c["slabs"]))
    re = c["re"] * rng.uniform(0.95, 1.05)
    h = H8(["--mesh", mesh, "--duct", "1", "--wall-model", "spalding", "--re", repr(re), "--alpha-u", "0.5",
            "--alpha-p", "0.3", "--amg-hierarchy", "cf", "--cf-interp", "exti", "--cf-theta", "0.25",
            "--amg-terminal", "1000", "--amg-smoother", "mcgs", "--amg-mcgs-order", "symmetric",
            "--pressure-solver", "pcg", "--p-rtol", "1e-3", "--p-atol", "1e-12", "--run-mode", "converge",
            "--max-outer", "1000", "--simple-tol", "1e-13", "--p-max", "600", "--verbose", "0",
            "--amg-precision", c["precision"]])
    # the third sample at y+ = 30 for the Blasius friction velocity, one
    # ray-traced Spalding point, the log-layer omega target on the wall faces
    y30 = 30.0 / (re * math.sqrt(0.3164 * re ** -0.25 / 8.0))
    h.turb_init(["--sst-wall-sample-scale", repr(y30 / (4.4084029504620439e-4 / 0.004)), "--sst-wall-sampling",
                 "ray_trace", "--sst-wall-active-points", "1", "--sst-wall-ray-local-adapt", "1",
                 "--sst-omega-wall-target", "trace_log"])
    h.wall_init(["--convection-form", "advective"])
    u0 = h.get("wall_u0", 3 * h.info["nv"]).reshape(-1, 3)
    s = {"h": h, "rest_p": np.zeros(h.info["cells"]), "u": [np.ascontiguousarray(u0[:, d]) for d in range(3)]}
    _turb_start(h, s)
    return s


@functools.lru_cache(maxsize=2)
def _laplacian(n):
    return p1.kuhn_p1_laplacian(n)


def prepare(case, seed):
    c, rng = case, np.random.default_rng(seed)
    s = {}
    if c["kind"] == "laminar":
        s = _laminar(c, rng)
    elif c["kind"] == "poisson":
        row, col, val = _laplacian(c["n"])
        order = "sweeps=2 order=forward" if c["smoother"] == "mcgs" else "sweeps=1 omega=0.7"
        s["S"] = System(row, col, val, f"precision={c['precision']} smoother={c['smoother']} {order}")
        s["b"] = p1.poisson_rhs(row.size - 1, seed=seed)
    elif c["kind"] == "komega":
        # the velocity of a short laminar run at the seed's Reynolds number
        h = H8(["--mesh", _pipe(c), "--re", repr(rng.uniform(10.0, 45.0)), "--p-rtol", "0.5"] + _BENCH + _converge(40))
        h.run()
        h.turb_init([])
        s["h"] = h
        _turb_start(h, s)
    elif c["kind"] == "sst":
        h = H8(["--mesh", _pipe(c), "--re", repr(rng.uniform(150.0, 250.0)), "--mom-sweeps", "20", "--mom-omega", "0.7",
                "--p-rtol", "1e-3"] + _BENCH + ["--alpha-u", "0.7", "--alpha-p", "0.3"] + _converge(c["its"]) +
               ["--amg-precision", c["precision"]])
        h.turb_init([])
        h.turb_couple(True)
        s = {"h": h, "rest_p": np.zeros(h.info["cells"]), "rest_u": np.zeros(h.info["nv"])}
        _turb_start(h, s)
    elif c["kind"] == "wall":
        s = _wall(c, rng)
    else:
        s["h"] = H8(["--mesh", _pipe(c)] + _BENCH + _converge(10))
        s["g"] = Gnn(s["h"], seed=1)
        s["g"].set_params(_gnn_params(rng))
        s["x"], s["t"] = _gnn_sample(s["g"].n, rng)
    s["case"] = c
    return s


def run(s):
    c = s["case"]
    if c["kind"] == "poisson":
        x, _ = s["S"].solve(s["b"], "fgmres", 1e-8, 30, 500)
        return {"x": x}
    if c["kind"] == "gnn":
        y = s["g"].forward(s["x"])
        grad, loss = s["g"].gradient(s["x"], s["t"])
        return {"y": y, "loss": float(loss), "grad": _gnn_split(grad)}
    h = s["h"]
    turb = c["kind"] in ("komega", "sst", "wall")
    if turb:
        h.set("k", s["k"])
        h.set("omega", s["omega"])
    if c["kind"] == "komega":
        for _ in range(c["steps"]):
            h.turb_step()
        return {"k": h.get("k", h.turb["ns"]), "omega": h.get("omega", h.turb["ns"])}
    h.set("p", s["rest_p"])
    for d in range(3):
        h.set(f"u{d}", s["u"][d] if "u" in s else s["rest_u"])
    if c["kind"] == "wall":
        h.run_window(1, c["its"])
    else:
        h.run()
    out = {f"u{d}": h.get(f"u{d}", h.info["nv"]) for d in range(3)}
    out["p"] = h.get("p", h.info["cells"])
    if turb:
        out["k"] = h.get("k", h.turb["ns"])
        out["omega"] = h.get("omega", h.turb["ns"])
    return out


# ----------------------------------------------------------------- work
def work(case):
    """Compulsory traffic of a pass.  Per cell of a tetrahedral mesh: 2.14
    free velocity DOFs, 35 momentum nonzeros, 66 P0 Schur nonzeros, 0.2
    vertices with 15 neighbours each."""
    c = case
    if c["kind"] == "poisson":
        n = (c["n"] + 1) ** 3
        nnz, its = 14.6 * n, 19
        s = {"fp64": 8, "fp32": 4, "bf16": 2}[c["precision"]]
        # a Krylov iteration: the operator and at least two smoothing passes,
        # two vectors of the basis written and one read again
        return {"bytes": its * (nnz * (12 + 2 * (s + 4)) + 48.0 * n), "flops": its * nnz * 6.0}
    nc = _cells(c)
    if c["kind"] == "gnn":
        # forward twice, backward once: the activations written and read once,
        # 2 M K N per product (K, N = 16 x 64, then four 128 x 64)
        return {"bytes": nc * (4 * (2 * 16 + 2) + 4 * 64 * 4 * 2.0 * 3), "flops": nc * 4 * 2.0 * (16 * 64 + 4 * 128 * 64)}
    nv, mom, fine, vert = 2.14 * nc, 35.0 * nc, 66.0 * nc, 0.2 * nc
    # one k-omega step: per equation the geometry and the two fields once, the
    # vertex operator written once and read in each of 20 sweeps
    step = 2 * (nc * (64 + 72 + 8) + nv * 24 + vert * (15 * 12 * 21 + 20 * 32))
    step_fl = 2 * (nc * 24 * (64 * 8 + 400.0) + 20 * vert * 15 * 2)
    if c["kind"] == "komega":
        return {"bytes": c["steps"] * step, "flops": c["steps"] * step_fl}
    s = 8 if c["precision"] == "fp64" else 4
    sweeps, its, block = (20, 20, 1) if c["kind"] == "sst" else (20, 40, 9) if c["kind"] == "wall" else (1, 3, 1)
    # one SIMPLE iteration: geometry and B, the momentum operator written once
    # and read in each sweep, the Schur values written once, and per Krylov
    # iteration the operator (in its factors B, rAU, B^T on the wall path) and
    # at least two smoothing passes
    op = fine * 12.0 if c["kind"] != "wall" else nc * (192 + 32 + 16) + nv * 24
    by = nc * (32 + 72 + 8 + 192) + (1 + sweeps) * (mom * (8.0 * block + 4) + 80 * nv) + fine * 12
    by += its * (op + 2 * fine * (s + 4) + 64 * nc)
    fl = (1 + sweeps) * mom * 6.0 * (3 if block == 9 else 1) + fine * 6 * 1.5 + its * fine * 6.0
    if c["kind"] != "laminar":
        by, fl = by + step, fl + step_fl
    return {"bytes": c["its"] * by, "flops": c["its"] * fl}


def tolerance(case):
    """About four times what the start shows between its own lane counts per
    row and others (sums in another order), rounded up; the sizes and numbers
    of iterations drawn vary it by a few times."""
    c = case
    if c["kind"] == "gnn":  # FP32 sums of BF16 products: a flipped rounding travels through five layers
        return {"rel": 2e-3, "max": 0.1}
    if c["kind"] == "poisson":  # 1e-11
        return {"rel": 1e-10}
    if c["kind"] == "komega":  # FP64, 2e-7: iterative wall fits that branch on rounding
        return {"rel": 1e-6, "max": 1e-5}
    fp64 = c["precision"] == "fp64"
    if c["kind"] == "sst":  # the same fits inside the loop: 3e-8 and 1e-7
        return {"rel": 2e-7, "max": 2e-6} if fp64 else {"rel": 5e-7, "max": 5e-6}
    if c["kind"] == "wall":  # 2e-14 and 8e-8
        return {"rel": 1e-12} if fp64 else {"rel": 4e-7, "max": 6e-6}
    return {"rel": 5e-12} if fp64 else {"rel": 7e-6, "max": 5e-5}  # 5e-13 and 1.7e-6


# ----------------------------------------------------------------- network
_IN, _HID, _LAYERS = 16, 64, 4
_SHAPES = [("W0", (_IN, _HID)), ("b0", (_HID,))]
for _l in range(_LAYERS):
    _SHAPES += [(f"W{_l + 1}", (2 * _HID, _HID)), (f"b{_l + 1}", (_HID,))]
_SHAPES += [("w", (_HID,)), ("b", (1,))]


def _gnn_params(rng):
    """Flat FP32 parameters: He-scaled weights, small biases, a small decoder."""
    out = []
    for name, shape in _SHAPES:
        scale = 0.05 if name[0] == "b" else 0.1 * math.sqrt(2.0 / _HID) if name == "w" else math.sqrt(1.0 / shape[0])
        out.append((rng.standard_normal(shape) * scale).ravel())
    return np.concatenate(out).astype(np.float32)


def _gnn_split(flat):
    out, o = {}, 0
    for name, shape in _SHAPES:
        n = int(np.prod(shape))
        out[name] = flat[o:o + n].reshape(shape)
        o += n
    return out


def _gnn_sample(n, rng):
    """Features of a SIMPLE iteration in their units (residuals and
    corrections of unit RMS, wall distance in [0, 1], one, two logarithms)
    and a target near the previous correction, at another level."""
    x = np.zeros((n, _IN), dtype=np.float32)
    x[:, :4] = rng.standard_normal((n, 4))
    x[:, 4] = rng.random(n)
    x[:, 5] = 1.0
    x[:, 6], x[:, 7] = rng.uniform(-1, 1, 2)
    return x, (x[:, 2] + 0.3 * rng.standard_normal(n) - 1.0).astype(np.float32)


# ----------------------------------------------------------------- 64 bits
def exact(case, seed):
    """The Poisson solution and the network in FP64.  The SIMPLE and k-omega
    paths have none: restated in plain numpy (assembly, coloured sweeps and
    the hierarchy's set-up in Python loops) one pass takes minutes."""
    c, rng = case, np.random.default_rng(seed)
    if c["kind"] == "poisson":
        return {"x": _exact_poisson(c["n"], seed)}
    if c["kind"] == "gnn":
        return _exact_gnn(c, rng)
    return None


def _exact_poisson(n, seed):
    """Conjugate gradients in FP64 to rounding on the edge form of the P1
    Laplacian of the Kuhn cube, with vertex 0 pinned to zero.

    Every tetrahedron is a monotone path of three axis edges; its gradients
    couple consecutive path vertices only, with vol / h^2 = h / 6.  An axis
    edge of a hex lies on two of its six paths when the other two
    coordinates agree (both low or both high), on one otherwise."""
    m, h = n + 1, 1.0 / n
    b = p1.poisson_rhs(m ** 3, seed=seed).reshape(m, m, m)
    pair = np.zeros((m, m))
    for a in (0, 1):
        for e in (0, 1):
            pair[a:n + a, e:n + e] += 2.0 if a == e else 1.0
    w = pair * (h / 6.0)  # weight of an axis edge by its two other coordinates

    def apply(x):
        y = np.zeros_like(x)
        for ax in range(3):
            xt, yt = np.moveaxis(x, ax, 0), np.moveaxis(y, ax, 0)
            f = w * (xt[1:] - xt[:-1])
            yt[1:] += f
            yt[:-1] -= f
        y[0, 0, 0] = 0.0
        return y

    diag = np.zeros((m, m, m))
    for ax in range(3):
        dt = np.moveaxis(diag, ax, 0)
        dt[1:] += w
        dt[:-1] += w
    x = np.zeros_like(b)
    r = b.copy()
    r[0, 0, 0] = 0.0
    z = r / diag
    p, rz, stop = z.copy(), float((r * z).sum()), 1e-14 * np.linalg.norm(b)
    for _ in range(4000):
        q = apply(p)
        alpha = rz / float((p * q).sum())
        x += alpha * p
        r -= alpha * q
        if np.linalg.norm(r) <= stop:
            break
        z = r / diag
        rz, old = float((r * z).sum()), rz
        p = z + (rz / old) * p
    return x.ravel()


def _exact_gnn(c, rng):
    tets = np.asarray(meshgen.straight_pipe(c["core"], c["ring"], c["slabs"])[1])
    n = tets.shape[0]
    faces = np.sort(np.concatenate([tets[:, [1, 2, 3]], tets[:, [0, 2, 3]], tets[:, [0, 1, 3]], tets[:, [0, 1, 2]]]), axis=1)
    cell = np.tile(np.arange(n), 4)
    order = np.lexsort((faces[:, 2], faces[:, 1], faces[:, 0]))
    f, cell = faces[order], cell[order]
    same = np.flatnonzero((f[1:] == f[:-1]).all(axis=1))
    i, j = np.concatenate([cell[same], cell[same + 1]]), np.concatenate([cell[same + 1], cell[same]])
    deg = np.bincount(i, minlength=n).astype(np.float64)
    order = np.argsort(i, kind="stable")
    i, j = i[order], j[order]
    start = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=n))])[:-1]

    def gather(v):  # sum over the neighbours of every cell (each has at least one)
        return np.add.reduceat(v[j], start, axis=0)

    P = {k: v.astype(np.float64) for k, v in _gnn_split(_gnn_params(rng)).items()}
    x, t = _gnn_sample(n, rng)
    x, t = x.astype(np.float64), t.astype(np.float64)
    Z0 = x @ P["W0"] + P["b0"]
    H, kept = np.maximum(Z0, 0.0), []
    for l in range(1, _LAYERS + 1):
        X = np.concatenate([H, gather(H) / deg[:, None]], axis=1)
        Z = X @ P[f"W{l}"] + P[f"b{l}"]
        H = H + np.maximum(Z, 0.0)
        kept.append((X, Z))
    y = H @ P["w"] + P["b"][0] + x[:, 2]
    d = y - t
    dy = 2.0 * d / n
    G = {"w": H.T @ dy, "b": np.array([dy.sum()])}
    dH = np.outer(dy, P["w"])
    for l in range(_LAYERS, 0, -1):
        X, Z = kept[l - 1]
        dZ = dH * (Z > 0)
        G[f"W{l}"], G[f"b{l}"] = X.T @ dZ, dZ.sum(axis=0)
        dX = dZ @ P[f"W{l}"].T
        dH = dH + dX[:, :_HID] + gather(dX[:, _HID:] / deg[:, None])
    dZ = dH * (Z0 > 0)
    G["W0"], G["b0"] = x.T @ dZ, dZ.sum(axis=0)
    return {"y": y, "loss": float(np.mean(d * d)), "grad": G}
