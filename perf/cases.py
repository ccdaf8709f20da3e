"""Workloads of the stencil library, as a user's program calls them, for timing.

Each case is one pass through the public Python binding (kgstencil.py) over
the C ABI: buffers are torch tensors on the device, handed over as device
pointers; the library's calls are asynchronous on its own stream, as in the
suite's host programs.

Families (the field "family" of a case):

* ``suite``      one launch of each of the twelve FP64 stencils at the
                 benchmark's sizes: 3D tests at nx x ny x ns, 2D tests at
                 nx x (ny*ns) (``./benchmark nx ny ns ...``).
* ``precision``  one lockstep step of the precision comparison: the FP64 field
                 converted to FP32 and BF16, laplacian and wave13pt in the
                 three types, per-plane gaussblur in two, and the error
                 statistics of the FP32 and BF16 results.
* ``vecmath``    the suite's non-stencil tests at the benchmark's sizes:
                 vecadd, matvec (nx x ny*ns) and sincos in FP64 and FP32, and
                 matmul C(nx,ns) += A(nx,ny) B(ny,ns).
* ``matmul``     matmul alone, at sizes of a dense product.
* ``life``       uint8 Game of Life, ``steps`` generations.
* ``poisson``    a Poisson solve from a zero guess to a relative residual of
                 1e-10.
* ``batch``      ``steps`` steps of many independent grids under one captured
                 graph, and the newest level of every grid brought to the host.
* ``serve``      a queue of jobs of mixed kinds, types, sizes and step counts
                 run by continuous batching, final fields on the host.
"""
from __future__ import annotations

import importlib.util
import math
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parents[1]
PKG = ROOT / "kernelgen-perf-tests_amd"


def _load(name):
    spec = importlib.util.spec_from_file_location(name, PKG / (name + ".py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


kg = _load("kgstencil")

# Stable coefficients (laplacian: amplification in [-1/2, 1]; wave13pt:
# fourth-order leapfrog with C = 3/32; gaussblur: sigma = 1; jacobi: the
# 9-point average), exact in FP32 and BF16 where the precision runs use them.
LAP = (0.25, 0.125)
WAVE = (1.296875, 0.125, -0.0078125)
GAUSS = tuple(math.exp(-r2 / 2.0) for r2 in (0, 1, 2, 4, 5, 8))
JAC = (0.0, 0.2, 0.05)
GRAD = (0.5, -0.25, 0.75)
UXX = (0.5, -0.3)
GSRB = (0.5, 0.05, -0.02, 0.03)
WHISP = (0.7, 0.3)
COEFS = {"laplacian": LAP, "wave13pt": WAVE, "gaussblur3": GAUSS, "jacobi2": JAC, "life2": ()}
# kind -> algorithmic arrays moved per point (read + written), operations per point
STENCILS = {"laplacian": (2, 8), "divergence": (4, 8), "gradient": (4, 6), "wave13pt": (3, 16),
            "uxx1": (6, 25), "tricubic": (5, 292), "tricubic2": (5, 292), "lapgsrb": (2, 28),
            "jacobi": (2, 11), "gaussblur": (2, 31), "whispering": (12, 40), "gameoflife": (2, 14)}

_ctx = None


def _context():
    """The program's one library context."""
    global _ctx
    if _ctx is None:
        _ctx = kg.Context(0)
    return _ctx


def listed():
    return [
        # a unit-test or coarse-level grid: launches and latency count
        {"name": "suite 64x32x32", "family": "suite", "nx": 64, "ny": 32, "ns": 32},
        # the benchmark's own sizes
        {"name": "suite 512x256x256", "family": "suite", "nx": 512, "ny": 256, "ns": 256},
        # a grid as a mesh generator leaves it: odd in every direction
        {"name": "suite 301x203x151", "family": "suite", "nx": 301, "ny": 203, "ns": 151},
        # the precision comparison at its own size, and on an odd grid
        {"name": "precision 512^3", "family": "precision", "nx": 512, "ny": 512, "ns": 512},
        {"name": "precision 333x257x131", "family": "precision", "nx": 333, "ny": 257, "ns": 131},
        # the benchmark's non-stencil rows
        {"name": "vecmath 512x256x256", "family": "vecmath", "nx": 512, "ny": 256, "ns": 256},
        # a dense product large enough to fill the chip
        {"name": "matmul 2048^3", "family": "matmul", "nx": 2048, "ny": 2048, "ns": 2048},
        # uint8 Life at its own size: ten generations between two pictures
        {"name": "life 8192^2", "family": "life", "nx": 8192, "ny": 8192, "steps": 10},
        # Poisson solves: a small one inside a time step, and the largest measured one
        {"name": "poisson 512", "family": "poisson", "n": 512, "vcycles": 2, "noalloc": False},
        {"name": "poisson 8192", "family": "poisson", "n": 8192, "vcycles": 2, "noalloc": False},
        # a parameter study: 40 grids of mixed size and kind, stepped together
        {"name": "batch 40 grids f32", "family": "batch", "grids": 40, "lo": 16, "hi": 128,
         "dtype": "f32", "steps": 400, "pick": 1},
        # a queue of 32 jobs, all present when the service starts
        {"name": "serve 32 jobs", "family": "serve", "jobs": 32, "vmin": 32 ** 3, "vmax": 128 ** 3,
         "smin": 10, "smax": 1000, "pick": 7},
    ]


def _log(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def _dims(rng, lo, nxm, nym, nsm):
    return {"nx": _log(rng, lo, nxm), "ny": _log(rng, lo, nym), "ns": _log(rng, lo, nsm)}


def draw(rng):
    family = rng.choice(["suite", "suite", "precision", "vecmath", "matmul", "life", "poisson",
                         "batch", "serve"])
    if family == "suite":
        return {"family": family, **_dims(rng, 24, 512, 256, 256)}
    if family == "precision":
        return {"family": family, **_dims(rng, 33, 512, 512, 512)}
    if family == "vecmath":
        return {"family": family, **_dims(rng, 48, 512, 256, 256)}
    if family == "matmul":
        return {"family": family, **_dims(rng, 128, 2048, 2048, 2048)}
    if family == "life":
        return {"family": family, "nx": _log(rng, 512, 8192), "ny": _log(rng, 512, 8192),
                "steps": rng.randint(1, 10)}
    if family == "poisson":
        n = 1 << rng.randint(6, 13)
        return {"family": family, "n": n, "vcycles": rng.randint(1, 3),
                "noalloc": n <= 1024 and rng.random() < 0.5}
    if family == "batch":
        return {"family": family, "grids": rng.randint(8, 40), "lo": 16,
                "hi": rng.randint(48, 128), "dtype": rng.choice(["f32", "f64"]),
                "steps": rng.randint(100, 400), "pick": rng.randrange(1 << 20)}
    return {"family": family, "jobs": rng.randint(4, 32), "vmin": 32 ** 3,
            "vmax": rng.randint(64, 128) ** 3, "smin": 10, "smax": rng.randint(100, 1000),
            "pick": rng.randrange(1 << 20)}


# ------------------------------------------------------------------ inputs
class _Inputs:
    """Seeded device tensors, uniform in [-1, 1) as the suite's real_rand()."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def uniform(self, n, lo=-1.0, hi=1.0):
        return torch.rand(n, generator=self.g, device="cuda", dtype=torch.float64).mul_(hi - lo).add_(lo)

    def cells(self, n):
        return torch.rand(n, generator=self.g, device="cuda", dtype=torch.float32) < 0.3


def _suite_inputs(case, seed):
    n = case["nx"] * case["ny"] * case["ns"]
    r = _Inputs(seed)
    a = {}
    a["laplacian"] = [r.uniform(n)]
    a["divergence"] = [r.uniform(n) for _ in range(3)]
    a["gradient"] = [r.uniform(n)]
    a["wave13pt"] = [r.uniform(n) for _ in range(2)]
    a["uxx1"] = [r.uniform(n), r.uniform(n, 1.0, 2.0)] + [r.uniform(n) for _ in range(3)]
    a["tricubic"] = [r.uniform(n) for _ in range(4)]
    a["tricubic2"] = [r.uniform(n) for _ in range(4)]
    a["lapgsrb"] = [r.uniform(n)]
    a["jacobi"] = [r.uniform(n)]
    a["gaussblur"] = [r.uniform(n)]
    # e (two components), h0, u_em0, ca, cb, da, db
    a["whispering"] = [r.uniform(2 * n)] + [r.uniform(n) for _ in range(6)]
    a["gameoflife"] = [r.cells(n).to(torch.float64)]
    return a


def _batch_grids(case):
    rng = np.random.default_rng(case["pick"])
    n = case["grids"]
    lo, hi = case["lo"], case["hi"]
    edges = np.exp(rng.uniform(np.log(lo), np.log(hi + 1), (n, 3)))
    edges = np.minimum(np.floor(edges), hi).astype(int)
    kinds = rng.choice(["laplacian", "gaussblur3", "wave13pt"], n)
    return [(str(k), tuple(int(v) for v in e)) for k, e in zip(kinds, edges)]


def _serve_jobs(case, seed):
    """Job mix of the serving runs: kind uniform, volume and steps
    log-uniform, FP64 or FP32; the 2D kinds as nx x (ny*ns) problems."""
    rng = np.random.default_rng(case["pick"])
    kinds = ["laplacian", "wave13pt", "gaussblur3", "jacobi2", "life2"]
    jobs = []
    for i in range(case["jobs"]):
        kind = kinds[int(rng.integers(0, 5))]
        v = math.exp(rng.uniform(math.log(case["vmin"]), math.log(case["vmax"])))
        s = (v / (512 * 256 * 256)) ** (1.0 / 3.0)
        nx, ny, ns = (max(3, round(e * s)) for e in (512, 256, 256))
        if kind in ("jacobi2", "life2"):
            ny, ns = ny * ns, 1
        steps = int(round(math.exp(rng.uniform(math.log(case["smin"]), math.log(case["smax"])))))
        jobs.append({"kind": kind, "dtype": kg.F64 if rng.random() < 0.5 else kg.F32,
                     "dims": (nx, ny, ns), "steps": steps, "coef": COEFS[kind],
                     "tol": 1e-8 if kind == "jacobi2" else 0.0, "arrival": 0.0,
                     "seed": 1000 * seed + i})
    return jobs


class _Grids:
    """A batch handle that is closed with the state that owns it."""

    def __init__(self, ctx):
        self.b = kg.Batch(ctx)

    def __del__(self):
        try:
            self.b.close()
        except Exception:
            pass


def prepare(case, seed):
    ctx = _context()
    fam = case["family"]
    st = {"case": case, "ctx": ctx}
    zeros = lambda n, dt=torch.float64: torch.zeros(n, dtype=dt, device="cuda")  # noqa: E731
    if fam == "suite":
        n = case["nx"] * case["ny"] * case["ns"]
        st["in"] = a = _suite_inputs(case, seed)
        nout = {"gradient": 3, "whispering": 0}
        st["out"] = {k: [zeros(n) for _ in range(nout.get(k, 1))] for k in a}
        # e's two buffers start equal (its border is never written); h1, u_em1
        st["out"]["whispering"] = [a["whispering"][0].clone(), zeros(n), zeros(n)]
    elif fam == "precision":
        n = case["nx"] * case["ny"] * case["ns"]
        r = _Inputs(seed)
        st["in"] = [r.uniform(n), r.uniform(n)]
        st["lo"] = [[torch.empty(n, dtype=dt, device="cuda") for _ in range(2)]
                    for dt in (torch.float32, torch.bfloat16)]
        st["out"] = {"lap": [zeros(n, dt) for dt in (torch.float64, torch.float32, torch.bfloat16)],
                     "wave": [zeros(n, dt) for dt in (torch.float64, torch.float32, torch.bfloat16)],
                     "gauss": [zeros(n, dt) for dt in (torch.float64, torch.float32)]}
    elif fam == "vecmath":
        nx, ny, ns = case["nx"], case["ny"], case["ns"]
        n = nx * ny * ns
        r = _Inputs(seed)
        d = {"p": r.uniform(n), "q": r.uniform(n), "x": r.uniform(nx)}
        st["f64"] = d
        st["f32"] = {k: v.to(torch.float32) for k, v in d.items()}
        st["out"] = {dt: {"add": zeros(n, ty), "mv": zeros(ny * ns, ty), "sc": zeros(n, ty)}
                     for dt, ty in (("f64", torch.float64), ("f32", torch.float32))}
        st["A"], st["B"], st["C"] = r.uniform(nx * ny), r.uniform(ny * ns), zeros(nx * ns)
    elif fam == "matmul":
        nx, ny, ns = case["nx"], case["ny"], case["ns"]
        r = _Inputs(seed)
        st["A"], st["B"], st["C"] = r.uniform(nx * ny), r.uniform(ny * ns), zeros(nx * ns)
    elif fam == "life":
        c = _Inputs(seed).cells(case["nx"] * case["ny"]).to(torch.uint8)
        st["in"] = c
        st["lv"] = [c.clone(), c.clone()]   # levels share the border
    elif fam == "poisson":
        N = case["n"] + 1
        st["f"], st["u"], st["u0"] = _poisson_f(case, seed), zeros(N * N), zeros(N * N)
    elif fam == "batch":
        st["hold"] = hold = _Grids(ctx)
        dt = kg.F32 if case["dtype"] == "f32" else kg.F64
        npd = np.float32 if case["dtype"] == "f32" else np.float64
        rng = np.random.default_rng(seed)
        st["ids"] = []
        for kind, (nx, ny, ns) in _batch_grids(case):
            gid = hold.b.add(kind, dt, (nx, ny, ns), COEFS[kind])
            nlev = kg.NLEV[kg.KINDS[kind]]
            a = rng.random(nx * ny * ns, dtype=npd) * 2 - 1   # every level starts alike
            for lev in range(nlev):
                hold.b.upload(gid, lev, a)
            st["ids"].append(gid)
    else:
        st["jobs"] = _serve_jobs(case, seed)
    torch.cuda.synchronize()
    return st


def _poisson_f(case, seed):
    N = case["n"] + 1
    f = _Inputs(seed).uniform(N * N)
    g = f.view(N, N)
    g[0], g[-1], g[:, 0], g[:, -1] = 0, 0, 0, 0
    return f


# -------------------------------------------------------------------- a pass
def run(st):
    case, ctx = st["case"], st["ctx"]
    p = torch.Tensor.data_ptr
    fam = case["family"]
    if fam == "suite":
        d3 = (case["nx"], case["ny"], case["ns"])
        d2 = (case["nx"], case["ny"] * case["ns"])
        a, o = st["in"], st["out"]
        ctx.call("laplacian", *d3, *LAP, p(a["laplacian"][0]), p(o["laplacian"][0]))
        ctx.call("divergence", *d3, *GRAD, p(o["divergence"][0]), *map(p, a["divergence"]))
        ctx.call("gradient", *d3, *GRAD, p(a["gradient"][0]), *map(p, o["gradient"]))
        ctx.call("wave13pt", *d3, *WAVE, *map(p, a["wave13pt"]), p(o["wave13pt"][0]))
        u0, d1, xx, xy, xz = map(p, a["uxx1"])
        ctx.call("uxx1", *d3, *UXX, u0, p(o["uxx1"][0]), d1, xx, xy, xz)
        for k in ("tricubic", "tricubic2"):
            u0, ta, tb, tc = map(p, a[k])
            ctx.call(k, *d3, u0, p(o[k][0]), ta, tb, tc)
        ctx.call("lapgsrb", *d3, *GSRB, p(a["lapgsrb"][0]), p(o["lapgsrb"][0]))
        ctx.call("jacobi", *d2, *JAC, p(a["jacobi"][0]), p(o["jacobi"][0]))
        ctx.call("gaussblur", *d2, *GAUSS, p(a["gaussblur"][0]), p(o["gaussblur"][0]))
        e, h0, um, ca, cb, da, db = map(p, a["whispering"])
        eo, h1, um1 = map(p, o["whispering"])
        ctx.call("whispering", *d2, *WHISP, e, eo, h0, h1, um, um1, ca, cb, da, db)
        ctx.call("gameoflife", *d2, p(a["gameoflife"][0]), p(o["gameoflife"][0]))
        return o
    if fam == "precision":
        d3 = (case["nx"], case["ny"], case["ns"])
        n = d3[0] * d3[1] * d3[2]
        w0, w1 = st["in"]
        f32, b16 = st["lo"]
        for code, lv in ((kg.F32, f32), (kg.BF16, b16)):
            for src, dst in zip((w0, w1), lv):
                ctx.call("convert", code, p(dst), kg.F64, p(src), n)
        o = st["out"]
        for q, (sfx, lv) in enumerate((("", (w0, w1)), ("_f32", f32), ("_bf16", b16))):
            ctx.call("laplacian" + sfx, *d3, *LAP, p(lv[0]), p(o["lap"][q]))
            ctx.call("wave13pt" + sfx, *d3, *WAVE, p(lv[0]), p(lv[1]), p(o["wave"][q]))
        ctx.call("gaussblur3_f64", *d3, *GAUSS, p(w0), p(o["gauss"][0]))
        ctx.call("gaussblur3_f32", *d3, *GAUSS, p(f32[0]), p(o["gauss"][1]))
        stats = {}
        for k in ("lap", "wave"):
            for q, code in ((1, kg.F32), (2, kg.BF16)):
                stats["%s%d" % (k, q)] = ctx.field_stats(_Ptr(o[k][q]), code, _Ptr(o[k][0]), kg.F64, n)
        return {**o, "stats": stats}
    if fam == "vecmath":
        nx, ny, ns = case["nx"], case["ny"], case["ns"]
        for dt, sfx in (("f64", ""), ("f32", "_f32")):
            d, o = st[dt], st["out"][dt]
            ctx.call("vecadd" + sfx, nx, ny, ns, p(d["p"]), p(d["q"]), p(o["add"]))
            ctx.call("matvec" + sfx, nx, ny * ns, p(d["p"]), p(d["x"]), p(o["mv"]))
            ctx.call("sincos" + sfx, nx, ny, ns, p(d["p"]), p(d["q"]), p(o["sc"]))
        ctx.call("matmul", nx, ny, ns, p(st["A"]), p(st["B"]), p(st["C"]))
        return {**st["out"], "C": st["C"]}
    if fam == "matmul":
        nx, ny, ns = case["nx"], case["ny"], case["ns"]
        ctx.call("matmul", nx, ny, ns, p(st["A"]), p(st["B"]), p(st["C"]))
        return st["C"]
    if fam == "life":
        nx, ny = case["nx"], case["ny"]
        src, lv = st["in"], st["lv"]
        for s in range(case["steps"]):
            ctx.call("life_u8", nx, ny, p(src), p(lv[s & 1]))
            src = lv[s & 1]
        return src
    if fam == "poisson":
        N = case["n"] + 1
        kg._check(ctx.lib, ctx.lib.kg_d2d(ctx.ptr, p(st["u"]), p(st["u0"]), N * N * 8), "kg_d2d")
        rep = kg.poisson_solve(ctx, case["n"], _Ptr(st["f"]), _Ptr(st["u"]), tol=1e-10, max_outer=30,
                               vcycles=case["vcycles"], noalloc=case["noalloc"])
        return {"u": st["u"], "outer": rep["outer"], "vcycles": rep["vcycles"], "levels": rep["levels"]}
    if fam == "batch":
        b = st["hold"].b
        b.step(case["steps"], graph=True)
        return [b.download(g) for g in st["ids"]]
    results, stats, fields = kg.serve(ctx, st["jobs"], 200 * 10 ** 9, 64, outputs=True)
    return {"fields": fields, "steps": np.array([r["steps_run"] for r in results]),
            "sums": np.array([r["checksum"] for r in results])}


class _Ptr:
    """A torch tensor where the binding takes a device array."""

    def __init__(self, t):
        self.ptr = t.data_ptr()
        self.shape = tuple(t.shape)


# --------------------------------------------------------------------- work
def work(case):
    """Bytes and operations of a pass: inputs read once, outputs written once
    (steps of a time loop each read and write their levels)."""
    fam = case["family"]
    if fam == "poisson":
        n = (case["n"] + 1) ** 2
        # f and the guess read, u written; about ten digits of a multigrid solve
        return {"bytes": 24 * n, "flops": 500 * n}
    if fam in ("batch", "serve"):
        b = f = 0
        if fam == "batch":
            todo = [(k, d, 4 if case["dtype"] == "f32" else 8, case["steps"]) for k, d in _batch_grids(case)]
        else:
            todo = [(j["kind"], j["dims"], 4 if j["dtype"] == kg.F32 else 8, j["steps"])
                    for j in _serve_jobs(case, 0)]
        name = {"gaussblur3": "gaussblur", "jacobi2": "jacobi", "life2": "gameoflife"}
        for kind, d, size, steps in todo:
            n = d[0] * d[1] * d[2]
            arrays, ops = STENCILS[name.get(kind, kind)]
            b += n * size * (arrays * steps + 1)
            f += n * ops * steps
        return {"bytes": b, "flops": f}
    nx, ny = case["nx"], case["ny"]
    if fam == "life":
        return {"bytes": 2 * nx * ny * case["steps"], "flops": 10 * nx * ny * case["steps"]}
    ns = case["ns"]
    n = nx * ny * ns
    if fam == "suite":
        return {"bytes": 8 * n * sum(a for a, _ in STENCILS.values()),
                "flops": n * sum(o for _, o in STENCILS.values())}
    if fam == "precision":
        # two fields converted (8 read, 6 written), lap 2 and wave 3 arrays in
        # 14 bytes, gaussblur 2 arrays in 12, statistics against both FP64 results
        return {"bytes": n * (2 * 14 + 2 * 14 + 3 * 14 + 2 * 12 + 2 * 14), "flops": n * (3 * 24 + 62 + 24)}
    if fam == "vecmath":
        mm = nx * ny + ny * ns + 2 * nx * ns
        return {"bytes": 12 * (7 * n + nx + ny * ns) + 8 * mm, "flops": n * 2 * (1 + 2 + 40) + 2 * n}
    return {"bytes": 8 * (nx * ny + ny * ns + 2 * nx * ns), "flops": 2 * n}


# -------------------------------------------------------------------- exact
def _shift3(w, lo, hi):
    """s(dx, dy, dz): the interior [lo, n-hi)^3 of w moved by an offset."""
    nz, ny, nx = w.shape

    def s(dx, dy=0, dz=0):
        return w[lo + dz:nz - hi + dz, lo + dy:ny - hi + dy, lo + dx:nx - hi + dx]
    return s


def _shift2(w, lo, hi):
    """The same on the last two axes (2D fields, or every plane of a 3D one)."""
    ny, nx = w.shape[-2:]

    def s(dx, dy=0):
        return w[..., lo + dy:ny - hi + dy, lo + dx:nx - hi + dx]
    return s


def _laplacian(w):
    s = _shift3(w, 1, 1)
    o = torch.zeros_like(w)
    o[1:-1, 1:-1, 1:-1] = LAP[0] * s(0) + LAP[1] * (s(1) + s(-1) + s(0, 1) + s(0, -1) + s(0, 0, 1) + s(0, 0, -1))
    return o


def _wave(w0, w1):
    s = _shift3(w1, 2, 2)
    ring = lambda d: (s(d) + s(-d) + s(0, d) + s(0, -d) + s(0, 0, d) + s(0, 0, -d))  # noqa: E731
    o = torch.zeros_like(w1)
    o[2:-2, 2:-2, 2:-2] = WAVE[0] * s(0) - w0[2:-2, 2:-2, 2:-2] + WAVE[1] * ring(1) + WAVE[2] * ring(2)
    return o


def _gauss(w):
    s0, s1, s2, s4, s5, s8 = GAUSS
    s = _shift2(w, 2, 2)
    tot = s0 * s(0)
    for c, offs in ((s1, ((1, 0), (0, 1))), (s2, ((1, 1), (1, -1))), (s4, ((2, 0), (0, 2))),
                    (s5, ((2, 1), (1, 2), (2, -1), (1, -2))), (s8, ((2, 2), (2, -2)))):
        for dx, dy in offs:
            tot = tot + c * (s(dx, dy) + s(-dx, -dy))
    o = torch.zeros_like(w)
    o[..., 2:-2, 2:-2] = tot / (s0 + 4 * (s1 + s2 + s4 + s8) + 8 * s5)
    return o


def _weights(t):
    return ((t * (t + 1) * (t + 2)) / 6, -(t - 1) * (t + 1) * (t + 2) / 2, (t - 1) * t * (t + 2) / 2,
            -(t - 1) * t * (t + 1) / 6)


def _tricubic(u, a, b, c, lo):
    s = _shift3(u, lo, 2)
    cut = lambda t: t[lo:-2, lo:-2, lo:-2]  # noqa: E731
    wa, wb, wc = _weights(cut(a)), _weights(cut(b)), _weights(cut(c))
    tot = torch.zeros_like(wa[0])
    for kk in range(4):
        for jj in range(4):
            row = sum(wa[ii] * s(ii - 1, jj - 1, kk - 1) for ii in range(4))
            tot += wb[jj] * wc[kk] * row
    o = torch.zeros_like(u)
    o[lo:-2, lo:-2, lo:-2] = tot
    return o


def _suite_exact(case, seed):
    nx, ny, ns = case["nx"], case["ny"], case["ns"]
    a = _suite_inputs(case, seed)
    v3 = {k: [t.view(ns, ny, nx) for t in v] for k, v in a.items()
          if k not in ("whispering", "jacobi", "gaussblur", "gameoflife")}
    v2 = lambda t: t.view(ny * ns, nx)  # noqa: E731
    o = {"laplacian": [_laplacian(v3["laplacian"][0])], "wave13pt": [_wave(*v3["wave13pt"])]}

    def put3(val, lo, hi):
        t = torch.zeros(ns, ny, nx, dtype=torch.float64, device="cuda")
        t[lo:ns - hi, lo:ny - hi, lo:nx - hi] = val
        return t
    sx, sy, sz = (_shift3(t, 1, 1) for t in v3["divergence"])
    al, be, ga = GRAD
    o["divergence"] = [put3(al * (sx(1) - sx(-1)) + be * (sy(0, 1) - sy(0, -1)) + ga * (sz(0, 0, 1) - sz(0, 0, -1)), 1, 1)]
    s = _shift3(v3["gradient"][0], 1, 1)
    o["gradient"] = [put3(al * (s(1) - s(-1)), 1, 1), put3(be * (s(0, 1) - s(0, -1)), 1, 1),
                     put3(ga * (s(0, 0, 1) - s(0, 0, -1)), 1, 1)]
    u0, d1, xx, xy, xz = (_shift3(t, 2, 1) for t in v3["uxx1"])
    d = (d1(0) + d1(0, -1) + d1(0, 0, -1) + d1(0, -1, -1)) / 4
    c1, c2 = UXX
    o["uxx1"] = [put3(u0(0) + (1.0 / nx / d) * (
        c1 * (xx(0) - xx(-1)) + c2 * (xx(1) - xx(-2)) + c1 * (xy(0) - xy(0, -1)) + c2 * (xy(0, 1) - xy(0, -2)) +
        c1 * (xz(0) - xz(0, 0, -1)) + c2 * (xz(0, 0, 1) - xz(0, 0, -2))), 2, 1)]
    o["tricubic"] = [_tricubic(*v3["tricubic"], 1)]
    o["tricubic2"] = [_tricubic(*v3["tricubic2"], 2)]
    s = _shift3(v3["lapgsrb"][0], 2, 2)
    face = lambda q: s(q) + s(-q) + s(0, q) + s(0, -q) + s(0, 0, q) + s(0, 0, -q)  # noqa: E731
    edge = sum(s(i, j, 0) + s(i, 0, j) + s(0, i, j) for i in (1, -1) for j in (1, -1))
    o["lapgsrb"] = [put3(GSRB[0] * s(0) + GSRB[1] * face(1) + GSRB[2] * edge + GSRB[3] * face(2), 2, 2)]
    w = v2(a["jacobi"][0])
    s = _shift2(w, 1, 1)
    t = torch.zeros_like(w)
    t[1:-1, 1:-1] = (JAC[0] * s(0) + JAC[1] * (s(1) + s(-1) + s(0, 1) + s(0, -1)) +
                     JAC[2] * (s(1, 1) + s(1, -1) + s(-1, 1) + s(-1, -1)))
    o["jacobi"] = [t]
    o["gaussblur"] = [_gauss(v2(a["gaussblur"][0]))]
    o["whispering"] = _whispering(a["whispering"], nx, ny * ns)
    w = v2(a["gameoflife"][0])
    s = _shift2(w, 1, 1)
    t = torch.zeros_like(w)
    L = sum(s(i, j) for i in (-1, 0, 1) for j in (-1, 0, 1) if i or j)
    t[1:-1, 1:-1] = 1 / (1 + (s(0) + L - 3) * (L - 3) * 1e20)
    o["gameoflife"] = [t]
    return {k: [t.reshape(-1) for t in v] for k, v in o.items()}


def _whispering(arrays, nx, ny):
    """The in-place sweep's values: where row j reads e0 of row j-1 (and e1 of
    column i-1), the sweep has updated it before, except on the border."""
    e, h0, um, ca, cb, da, db = arrays
    n = nx * ny
    e0, e1 = e[:n].view(ny, nx), e[n:].view(ny, nx)
    h, um, ca, cb, da, db = (t.view(ny, nx) for t in (h0, um, ca, cb, da, db))
    c, up, lf = (slice(1, -1), slice(1, -1)), (slice(0, -2), slice(1, -1)), (slice(1, -1), slice(0, -2))
    n0 = ca[c] * e0[c] + cb[c] * (h[2:, 1:-1] - h[c])
    n1 = ca[c] * e1[c] - cb[c] * (h[1:-1, 2:] - h[c])
    dy, dx = h[c] - h[up], h[c] - h[lf]
    ey, ex = ca[up] * e0[up] + cb[up] * dy, ca[lf] * e1[lf] - cb[lf] * dx
    ey[0], ex[:, 0] = e0[up][0], e1[lf][:, 0]
    ey, ex = ca[up] * ey + cb[up] * dy, ca[lf] * ex - cb[lf] * dx
    hn = da[c] * h[c] + db[c] * (n0 - ey + ex - n1)
    eo = e.clone()
    eo[:n].view(ny, nx)[c] = n0
    eo[n:].view(ny, nx)[c] = n1
    h1, u1 = torch.zeros_like(h), torch.zeros_like(h)
    h1[c] = hn
    u1[c] = um[c] + 0.5 * (hn * hn / WHISP[0] + WHISP[1] * (n0 * n0 + n1 * n1))
    return [eo, h1, u1]


def _life(c):
    c = c.clone()
    b = c[1:-1, 1:-1]
    k = sum(c[1 + j:c.shape[0] - 1 + j, 1 + i:c.shape[1] - 1 + i] for i in (-1, 0, 1) for j in (-1, 0, 1) if i or j)
    b.copy_(((k == 3) | ((b != 0) & (k == 2))).to(torch.uint8))
    return c


def _sines(x):
    """Sine transform along the last axis (values at 1 .. m of 0 .. m+1)."""
    m = x.shape[-1]
    z = torch.zeros(*x.shape[:-1], 1, dtype=x.dtype, device=x.device)
    return -torch.fft.rfft(torch.cat([z, x, z, -x.flip(-1)], -1))[..., 1:m + 1].imag


def _poisson_exact(case, seed):
    n = case["n"]
    f = _poisson_f(case, seed).view(n + 1, n + 1)[1:-1, 1:-1]
    cs = torch.cos(torch.arange(1, n, device="cuda", dtype=torch.float64) * math.pi / n)
    t = _sines(_sines(f).T.contiguous())
    t /= (20 - 8 * (cs[:, None] + cs[None, :]) - 4 * cs[:, None] * cs[None, :]) * (n * n / 6.0)
    u = torch.zeros(n + 1, n + 1, dtype=torch.float64, device="cuda")
    u[1:-1, 1:-1] = _sines(_sines(t).T.contiguous()) / (4.0 * n * n)
    return {"u": u.reshape(-1), "outer": None, "vcycles": None, "levels": None}


def exact(case, seed):
    fam = case["family"]
    if fam == "suite":
        return _suite_exact(case, seed)
    if fam == "precision":
        nx, ny, ns = case["nx"], case["ny"], case["ns"]
        r = _Inputs(seed)
        n = nx * ny * ns
        w = [r.uniform(n).view(ns, ny, nx), r.uniform(n).view(ns, ny, nx)]
        o = {"lap": [], "wave": [], "gauss": []}
        for dt in (torch.float64, torch.float32, torch.bfloat16):
            a, b = (t.to(torch.float32).to(dt).double() if dt == torch.bfloat16 else t.to(dt).double() for t in w)
            o["lap"].append(_laplacian(a).reshape(-1))
            o["wave"].append(_wave(a, b).reshape(-1))
            if dt != torch.bfloat16:
                o["gauss"].append(_gauss(a).reshape(-1))
        # the statistics are those of the rounded results: no value of their own
        return {**o, "stats": None}
    if fam == "vecmath":
        nx, ny, ns = case["nx"], case["ny"], case["ns"]
        st = prepare(case, seed)
        o = {}
        for dt in ("f64", "f32"):
            d = {k: v.double() for k, v in st[dt].items()}
            o[dt] = {"add": d["p"] + d["q"], "mv": (d["p"].view(ny * ns, nx) * d["x"]).sum(1),
                     "sc": torch.sin(d["p"]) + torch.cos(d["q"])}
        return {**o, "C": (st["B"].view(ns, ny) @ st["A"].view(ny, nx)).reshape(-1)}
    if fam == "matmul":
        nx, ny, ns = case["nx"], case["ny"], case["ns"]
        st = prepare(case, seed)
        return (st["B"].view(ns, ny) @ st["A"].view(ny, nx)).reshape(-1)
    if fam == "life":
        c = _Inputs(seed).cells(case["nx"] * case["ny"]).to(torch.uint8).view(case["ny"], case["nx"])
        for _ in range(case["steps"]):
            c = _life(c)
        return c.reshape(-1)
    if fam == "poisson":
        return _poisson_exact(case, seed)
    return None   # hundreds of steps of many grids: too long this way
