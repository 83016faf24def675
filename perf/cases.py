"""Performance cases of the framework: what its users run, through its public entry points.

listed() holds the cases that are timed, draw() gives further ones of the same
ranges.  A case is a dict of plain values; prepare() makes what a program has
in hand before the call (fields or matrices in device memory, options, a
plan), run() is one pass through a public entry point and returns its whole
result, work() what the pass cannot do without, exact() the same result in 64
bits from plain torch.

Five families, by "kind":
  j3d    perks_amd.j3d_device: Jacobi steps on a 3D field in device memory
  j2d    perks_amd.jacobi2d_device: the same in 2D
  host   perks_amd.j3d_iterative: the drop-in call, host arrays in and out
  batch  perks_amd.BatchPlan.run: many uneven 2D grids, one replayed plan
  cg     perks_amd.cg_solve: a Poisson system solved to a tolerance
"""
import math
import random

import numpy as np
import torch

import perks_amd as P

DEV = "cuda"
TORCH = {"f64": torch.float64, "f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f64": 8, "f32": 4, "f16": 2, "bf16": 2}
LARGEST_J3D = 512**3 * 1000    # cell updates of the largest 3D solve
LARGEST_J2D = 8192**2 * 500    # of the largest 2D solve
MAX_ITER = 4000                # of a linear solve: several times what any of them takes
SHAPES_3D = ("3d7pt", "3d13pt", "3d17pt", "3d27pt", "poisson")
SHAPES_2D = ("2d5pt", "2ds9pt", "2d13pt", "2d9pt", "2d25pt")


def listed():
    return [
        # The headline solve: heat-like 7-point star in FP64, equal neighbour
        # weights, fixed zero halo, a thousand steps in one call.
        dict(name="j3d7_f64_512", kind="j3d", shape="3d7pt", dtype="f64", boundary="zero", method="persistent",
             weights="diffusion", rounding="nearest", nz=512, ny=512, nx=512, steps=1000),
        # A simulation's ordinary domain: odd sides, replicated edges (the
        # library's default boundary), weights of an anisotropic grid, FP32.
        dict(name="j3d7_f32_ragged_clamp", kind="j3d", shape="3d7pt", dtype="f32", boundary="clamp",
             method="persistent", weights="seeded", rounding="nearest", nz=301, ny=397, nx=455, steps=100),
        # A small domain advanced a few steps between other work: the call's
        # fixed costs and the grid barrier.
        dict(name="j3d7_f64_64", kind="j3d", shape="3d7pt", dtype="f64", boundary="zero", method="persistent",
             weights="diffusion", rounding="nearest", nz=64, ny=64, nx=64, steps=20),
        # Half the memory for the same field: BF16 storage, unbiased rounding.
        dict(name="j3d7_bf16sr_512", kind="j3d", shape="3d7pt", dtype="bf16", boundary="zero", method="persistent",
             weights="diffusion", rounding="stochastic", nz=512, ny=512, nx=512, steps=200),
        # A dense 3D shape: the 27-point box with weights of its own.
        dict(name="j3d27_f64_256", kind="j3d", shape="3d27pt", dtype="f64", boundary="clamp", method="persistent",
             weights="seeded", rounding="nearest", nz=256, ny=256, nx=256, steps=50),
        # The drop-in call of a program that keeps its field in host memory:
        # the shape's own weights, copies in and out, a few steps.
        dict(name="host_j3d7_f32_256", kind="host", shape="3d7pt", dtype="f32", boundary="clamp",
             method="persistent", nz=256, ny=256, nx=256, steps=10),
        # The 2D parity configuration: one launch per step, FP64, 5-point star.
        dict(name="j2d5_f64_2048_plain", kind="j2d", shape="2d5pt", dtype="f64", boundary="zero", method="plain",
             weights="diffusion", rounding="nearest", ny=2048, nx=2048, steps=100),
        # A large 2D solve: radius-1 box, seeded normalised weights, FP32.
        dict(name="j2d9_f32_8192", kind="j2d", shape="2d9pt", dtype="f32", boundary="zero", method="persistent",
             weights="seeded", rounding="nearest", ny=8192, nx=8192, steps=500),
        # 16-bit storage in 2D, radius-2 box, odd sides.
        dict(name="j2d25_f16_ragged", kind="j2d", shape="2d25pt", dtype="f16", boundary="zero", method="persistent",
             weights="seeded", rounding="nearest", ny=5003, nx=7001, steps=60),
        # Many independent uneven grids, refilled and replayed through a plan.
        dict(name="batch5_f32_512grids", kind="batch", shape="2d5pt", dtype="f32", grids=512, low=64, high=1024,
             min_steps=50, max_steps=500),
        # A linear solve: Poisson matrix in CSR, FP64, to a tight tolerance.
        dict(name="cg_csr_f64_256", kind="cg", fmt="csr", precision="f64", nx=256, ny=256, nz=256, tol=1e-10),
        # A small solve: DIA, FP32 inner iterations inside FP64 refinement;
        # what an iteration costs when the problem does not fill the chip.
        dict(name="cg_dia_refine_64", kind="cg", fmt="dia", precision="f32_refine", nx=64, ny=64, nz=64, tol=1e-10),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _fewer(c):
    """16-bit fields lose meaning over many steps, soonest in BF16 rounded to nearest."""
    return {8: 1, 4: 1, 2: 10 if (c["dtype"], c["rounding"]) == ("bf16", "nearest") else 5}[BYTES[c["dtype"]]]


def _drift_limit(c):
    """Unequal weights carry the field along; through a zero halo it leaves a small domain after a while."""
    short = min(c.get("nz", 1 << 20), c["ny"], c["nx"])
    return 2 * short if (c["weights"], c["boundary"]) == ("seeded", "zero") else 1 << 20


def draw(rng):
    kind = rng.choice(("j3d", "j3d", "j3d", "host", "j2d", "j2d", "batch", "cg", "cg"))
    if kind == "j3d":
        dtype = rng.choice(("f64", "f64", "f32", "f32", "bf16", "f16"))
        c = dict(kind=kind, shape=rng.choice(SHAPES_3D[:1] * 4 + SHAPES_3D), dtype=dtype,
                 boundary=rng.choice(("zero", "clamp")), method=rng.choice(("persistent", "persistent", "plain")),
                 weights=rng.choice(("diffusion", "seeded")),
                 rounding=rng.choice(("nearest", "stochastic")) if dtype in ("f16", "bf16") else "nearest",
                 nz=_log(rng, 48, 512), ny=_log(rng, 48, 512), nx=_log(rng, 48, 512))
        if dtype in ("f16", "bf16"):
            c["nx"] += c["nx"] % 2  # the per-step 16-bit kernel takes even widths
        # dense shapes cost more a step
        few = (1 if c["shape"] == "3d7pt" else 5) * _fewer(c)
        most = min(1000 // few, LARGEST_J3D // few // (c["nz"] * c["ny"] * c["nx"]), _drift_limit(c))
        c["steps"] = _log(rng, 5, max(6, most))
    elif kind == "host":
        c = dict(kind=kind, shape="3d7pt", dtype=rng.choice(("f64", "f32")), boundary=rng.choice(("zero", "clamp")),
                 method="persistent", nz=_log(rng, 32, 256), ny=_log(rng, 32, 256), nx=_log(rng, 32, 256),
                 steps=rng.randint(3, 20))
    elif kind == "j2d":
        dtype = rng.choice(("f64", "f32", "f32", "bf16", "f16"))
        c = dict(kind=kind, shape=rng.choice(SHAPES_2D), dtype=dtype, boundary=rng.choice(("zero", "clamp")),
                 method=rng.choice(("persistent", "persistent", "plain")), weights=rng.choice(("diffusion", "seeded")),
                 rounding=rng.choice(("nearest", "stochastic")) if dtype in ("f16", "bf16") else "nearest",
                 ny=_log(rng, 64, 8192), nx=_log(rng, 64, 8192))
        few = (2 if c["shape"] == "2d25pt" else 1) * _fewer(c)
        most = min(500 // few, LARGEST_J2D // few // (c["ny"] * c["nx"]), _drift_limit(c))
        c["steps"] = _log(rng, 10, max(11, most))
    elif kind == "batch":
        c = dict(kind=kind, shape=rng.choice(("2d5pt", "2d9pt")), dtype="f32", grids=_log(rng, 16, 320),
                 low=rng.choice((48, 64, 96)), high=rng.choice((512, 768, 1000)), min_steps=rng.randint(20, 50),
                 max_steps=rng.randint(200, 450))
    else:
        c = dict(kind=kind, fmt=rng.choice(("csr", "dia")), precision=rng.choice(("f64", "f64", "f32_refine")),
                 nx=_log(rng, 20, 240), ny=_log(rng, 20, 240), nz=_log(rng, 20, 240),
                 tol=rng.choice((1e-8, 1e-10)))
    return c


# ---- inputs ---------------------------------------------------------------------
def _weights(case, seed):
    """One weight per group of the shape; over its points they sum to 1, so the
    field stays bounded over any number of steps."""
    si = P.shape_info(case["shape"])
    if case["weights"] == "diffusion":  # equal neighbours; the centre heavier in the 7-point star
        if case["shape"] == "3d7pt":
            return [0.1] * 6 + [0.4]
        raw = [1.0] * len(si.coef)
    else:  # uniform in [0, 1)
        rng = random.Random(seed * 1009 + 17)
        raw = [rng.random() for _ in si.coef]
    total = sum(w * n for w, n in zip(raw, si.npts))
    return [w / total for w in raw]


def _field(shape, dtype, seed):
    """Uniform in [0, 1), rounded to the storage type."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return torch.rand(shape, generator=g, dtype=torch.float64 if dtype == "f64" else torch.float32,
                      device=DEV).to(TORCH[dtype])


def _host_field(case, seed):
    return np.random.default_rng(seed).random((case["nz"], case["ny"], case["nx"]),
                                              dtype=np.float64 if case["dtype"] == "f64" else np.float32)


def _grids(case):
    """Sides log-uniform and not square, step counts uniform; the plan's shape, the same for every input."""
    rng = random.Random(case["grids"])
    return [(_log(rng, case["low"], case["high"]), _log(rng, case["low"], case["high"]),
             rng.randint(case["min_steps"], case["max_steps"])) for _ in range(case["grids"])]


def _rhs(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    n = case["nx"] * case["ny"] * case["nz"]
    return torch.rand(n, generator=g, dtype=torch.float64, device=DEV) * 2 - 1


class State:
    pass


def prepare(case, seed):
    s = State()
    s.case = case
    kind = case["kind"]
    if kind in ("j3d", "j2d"):
        s.dims = (case["nz"], case["ny"], case["nx"]) if kind == "j3d" else (case["ny"], case["nx"])
        s.a = _field(s.dims, case["dtype"], seed)
        s.b = torch.zeros_like(s.a)
        s.opts = P.make_opts(case["shape"], case["boundary"], case["method"], coefs=_weights(case, seed),
                             rounding=case["rounding"], round_seed=seed)
    elif kind == "host":
        s.h_in = _host_field(case, seed)
        s.h_out = np.empty_like(s.h_in)
    elif kind == "batch":
        s.sizes = _grids(case)
        total = sum(h * w for h, w, _ in s.sizes)
        s.inputs = _field(total, case["dtype"], seed)
        s.fields = torch.empty_like(s.inputs)
        s.spare = torch.zeros_like(s.inputs)
        grids, at = [], 0
        for h, w, steps in s.sizes:
            grids.append((s.fields[at:at + h * w], s.spare[at:at + h * w], h, w, steps))
            at += h * w
        s.plan = P.BatchPlan(grids, dtype=case["dtype"], autotune=True,
                             opts=P.make_opts(case["shape"], "zero", "persistent", coefs=_batch_weights(case)))
        s.results = [b if in_b else a for (a, b, _, _, _), in_b in zip(grids, s.plan.result_in_b)]
    else:
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        s.n = nx * ny * nz
        s.b = _rhs(case, seed)
        s.x = torch.zeros_like(s.b)
        if case["fmt"] == "csr":
            nnz = P.poisson7_nnz(nx, ny, nz)
            s.matrix = dict(rowptr=torch.empty(s.n + 1, dtype=torch.int32, device=DEV),
                            col=torch.empty(nnz, dtype=torch.int32, device=DEV),
                            val=torch.empty(nnz, dtype=torch.float64, device=DEV))
            P.poisson7_csr(nx, ny, nz, **s.matrix)
            s.matrix["nnz"] = nnz
        else:
            val = torch.empty(7 * s.n, dtype=torch.float64, device=DEV)
            s.matrix = dict(offsets=P.poisson7_dia(nx, ny, nz, val), val=val)
    return s


def run(s):
    case = s.case
    kind = case["kind"]
    if kind in ("j3d", "j2d"):
        # a time loop: the result is the next call's input
        call = P.j3d_device if kind == "j3d" else P.jacobi2d_device
        rep = call(s.a, s.b, *s.dims, case["steps"], dtype=case["dtype"], opts=s.opts)
        if rep.result_in_b:
            s.a, s.b = s.b, s.a
        return s.a
    if kind == "host":
        rc = P.j3d_iterative(s.h_in, case["nz"], case["ny"], case["nx"], s.h_out, iteration=case["steps"],
                             shape=case["shape"], boundary=case["boundary"], method=case["method"])
        P.check(rc, "j3d_iterative")
        return s.h_out
    if kind == "batch":
        s.fields.copy_(s.inputs)  # new inputs into the plan's buffers
        s.plan.run()
        return torch.cat(s.results)
    s.x.zero_()
    res = P.cg_solve(case["fmt"], s.n, s.b, s.x, tol=case["tol"], precision=case["precision"], x0_is_zero=True,
                     max_iter=MAX_ITER, **s.matrix)
    history = np.zeros(MAX_ITER + 1)
    history[:len(res.history)] = res.history
    return {"x": s.x, "residual_history": history, "iterations": res.iterations}


# ---- what a pass cannot do without --------------------------------------------------
def work(case):
    """Bytes: every input read once and every output written once (CG: the
    matrix and six vectors once an iteration, they do not fit on the chip at
    the sizes that matter).  Operations: every product and sum of the updates."""
    kind = case["kind"]
    if kind == "cg":
        n = case["nx"] * case["ny"] * case["nz"]
        nnz = P.poisson7_nnz(case["nx"], case["ny"], case["nz"])
        # iterations grow with the longest side (about 4 per point at 1e-10)
        iters = 4 * max(case["nx"], case["ny"], case["nz"]) * (1.0 if case["tol"] < 1e-9 else 0.8)
        v = 8 if case["precision"] == "f64" else 4
        matrix = nnz * (v + 4) + 4 * (n + 1) if case["fmt"] == "csr" else 7 * n * v
        return {"bytes": iters * (matrix + 6 * n * v), "flops": iters * (2.0 * nnz + 12.0 * n)}
    si = P.shape_info(case["shape"])
    per_cell = sum(si.npts) - len(si.npts) + 2 * len(si.coef) - 1  # sums in the groups, products, sums of groups
    if kind == "batch":
        sizes = _grids(case)
        cells, updates = sum(h * w for h, w, _ in sizes), sum(h * w * t for h, w, t in sizes)
    else:
        cells = case.get("nz", 1) * case["ny"] * case["nx"]
        updates = cells * case["steps"]
    return {"bytes": 2.0 * cells * BYTES[case["dtype"]], "flops": float(updates) * per_cell}


# ---- the results in 64 bits ------------------------------------------------------------
def _steps64(u, points, radius, boundary, steps):
    """`steps` Jacobi steps of u: points is a list of (offsets, weight)."""
    d = u.dim()
    a = torch.zeros([n + 2 * radius for n in u.shape], dtype=torch.float64, device=u.device)
    b = torch.zeros_like(a)
    inner = tuple(slice(radius, radius + n) for n in u.shape)
    a[inner] = u
    for _ in range(steps):
        if boundary == "clamp":
            for axis in range(d):
                n = u.shape[axis]
                a.narrow(axis, 0, radius).copy_(a.narrow(axis, radius, 1).expand_as(a.narrow(axis, 0, radius)))
                a.narrow(axis, radius + n, radius).copy_(
                    a.narrow(axis, radius + n - 1, 1).expand_as(a.narrow(axis, 0, radius)))
        out = b[inner]
        for k, (off, w) in enumerate(points):
            src = a[tuple(slice(radius + o, radius + o + n) for o, n in zip(off, u.shape))]
            if k == 0:
                torch.mul(src, w, out=out)
            else:
                out.add_(src, alpha=w)
        a, b = b, a
    return a[inner].contiguous()


def _points(shape, weights):
    si = P.shape_info(shape)
    return [(off[3 - si.dims:], w) for pts, w in zip(si.offsets, weights) for off in pts], si.radius


def _batch_weights(case):
    n = len(P.shape_info(case["shape"]).coef)
    return [1.0 / n] * n


def _sines(n):
    """The eigenvectors of the second difference with fixed zero ends, and the cosines of their angles."""
    j = torch.arange(1, n + 1, dtype=torch.float64, device=DEV)
    k = torch.remainder(torch.outer(j, j), 2 * (n + 1))  # whole numbers: the angles stay exact
    return math.sqrt(2.0 / (n + 1)) * torch.sin(k * (math.pi / (n + 1))), torch.cos(j * (math.pi / (n + 1)))


def _batch64(case, seed):
    """Equal weights and a zero halo: the sine transform turns every step into one product."""
    flat = _field(sum(h * w for h, w, _ in _grids(case)), case["dtype"], seed).double()
    out, at, w0 = [], 0, _batch_weights(case)[0]
    for h, w, steps in _grids(case):
        u = flat[at:at + h * w].view(h, w)
        at += h * w
        sy, cy = _sines(h)
        sx, cx = _sines(w)
        if case["shape"] == "2d5pt":
            gain = w0 * (1 + 2 * cy[:, None] + 2 * cx[None, :])
        else:
            gain = w0 * (1 + 2 * cy[:, None]) * (1 + 2 * cx[None, :])
        out.append((sy @ ((sy @ u @ sx) * gain.pow(steps)) @ sx).reshape(-1))
    return torch.cat(out)


def _poisson64(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    (sx, cx), (sy, cy), (sz, cz) = _sines(nx), _sines(ny), _sines(nz)

    def transform(v):
        v = (v.reshape(-1, nx) @ sx).view(nz, ny, nx)
        v = (v.transpose(1, 2).reshape(-1, ny) @ sy).view(nz, nx, ny).transpose(1, 2).contiguous()
        return (sz @ v.view(nz, -1)).view(nz, ny, nx)

    eig = 6 - 2 * cz[:, None, None] - 2 * cy[None, :, None] - 2 * cx[None, None, :]
    return transform(transform(_rhs(case, seed)) / eig).reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return _batch64(case, seed)
    if kind == "cg":
        return {"x": _poisson64(case, seed), "residual_history": None, "iterations": None}
    if kind == "host":
        u = torch.from_numpy(_host_field(case, seed)).to(DEV).double()
        points, radius = _points(case["shape"], P.shape_info(case["shape"]).coef)
    else:
        dims = (case["nz"], case["ny"], case["nx"]) if kind == "j3d" else (case["ny"], case["nx"])
        u = _field(dims, case["dtype"], seed).double()
        points, radius = _points(case["shape"], _weights(case, seed))
    out = _steps64(u, points, radius, case["boundary"], case["steps"])
    return out.cpu().numpy() if kind == "host" else out
