"""Performance cases: the work a user of fastqsl_amd has it do.

Each case is one pass through a public entry point with its inputs resident
on the GPU (a field handle, seeds, a planned batch, the notebooks' arrays).
Fields and seeds are made from the seed alone: random sub-surface point
sources (the repository's multipole benchmark field, other sources for each
seed), with a flux rope added for the volume case, and seed planes whose edges
move by up to a tenth of a cell.

Kinds:
  lines      a handful of field lines traced by hand (latency of one call)
  map        ``scott_qmap`` of a constant-z seed grid
  plane      ``scott_qmap_plane``: an oblique plane through three points
  cube       ``scott_qcube``: Q on every sample of a 3-D box
  batch      ``ScottBatch.run``: uneven maps over resident fields
  neighbour  ``neighbour_qmap``: footpoint differences with pseudo lines
  stretch    ``trace_plain`` on a stretched grid
  twist      ``trace_scott`` with the twist number
  dropin     the reference-shaped call on the notebooks' own arrays
  snapshot   a new field: layouts built, one map traced, field released
"""
import math

import numpy as np
import torch

import fastqsl_amd as fq
from fastqsl_amd import postproc, qmap
from fastqsl_amd.batch import ScottBatch
from fastqsl_amd.trace import PLAIN_OUTPUTS, SCOTT_OUTPUTS

DEV = "cuda"


# ------------------------------------------------------------------- cases
def listed():
    return [
        # a user clicks a few seed points to look at single field lines
        dict(name="lines_64", kind="lines", n=64, nx=64, ny=64, nz=64, method="rkf45", tol=1e-6, precision="fp32c"),
        # the parity configuration: fixed-step RK4 on a small float64 field
        dict(name="map_rk4_fp64_256", kind="map", nu=256, nv=256, nx=64, ny=64, nz=64, method="rk4", tol=0.0,
             precision="fp64"),
        # the headline configuration: adaptive map of a full magnetogram
        dict(name="map_1024", kind="map", nu=1024, nv=1024, nx=256, ny=256, nz=256, method="rkf45", tol=1e-6,
             precision="fp32c"),
        # a vertical cut through a box that is no power of two, odd pixel counts
        dict(name="plane_777x333", kind="plane", nu=777, nv=333, nx=320, ny=200, nz=161, method="rkf45", tol=1e-5,
             precision="fp32c"),
        # 3-D Q of a flux rope, every second node across the rope: the largest job
        dict(name="cube_512x128x128", kind="cube", sx=512, sy=128, sz=128, nx=512, ny=256, nz=256, method="rkf45",
             tol=1e-6, precision="fp32c"),
        # a queue of uneven requests, RK4 and RKF45 in turn, over three fields
        dict(name="batch_12", kind="batch", requests=12, side_lo=64, side_hi=700, nx=256, ny=256, nz=192,
             precision="fp32c"),
        # the notebooks' usual map: footpoint differences and pseudo lines
        dict(name="neighbour_1024", kind="neighbour", nu=1024, nv=1024, nx=256, ny=256, nz=256, method="rkf45",
             precision="fp32c"),
        # a quick look at a region: a small odd map on a small field
        dict(name="neighbour_233x191", kind="neighbour", nu=233, nv=191, nx=128, ny=130, nz=96, method="rkf45",
             precision="fp32c"),
        # simulation output on a non-uniform grid
        dict(name="stretch_1024", kind="stretch", nu=1024, nv=1024, nx=256, ny=256, nz=256, precision="fp32c"),
        # Q and twist of an active region
        dict(name="twist_512", kind="twist", nu=512, nv=512, nx=256, ny=256, nz=256, tol=1e-6, precision="fp32c"),
        # a reference notebook run unchanged
        dict(name="dropin_384", kind="dropin", nu=384, nv=384, nx=256, ny=256, nz=256, tracer="scott"),
        # one step of a time series: every snapshot is a new field
        dict(name="snapshot_320", kind="snapshot", nu=256, nv=256, nx=320, ny=320, nz=256, tol=1e-6,
             precision="fp32c"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi):
    return dict(nx=_log_int(rng, lo, hi), ny=_log_int(rng, lo, hi), nz=_log_int(rng, lo, hi))


def draw(rng):
    kind = rng.choice(["lines", "map", "map", "plane", "cube", "batch", "neighbour", "neighbour", "stretch", "twist",
                       "dropin", "snapshot"])
    tol = 10.0 ** rng.uniform(-7.0, -5.0)
    method = rng.choice(["rkf45", "rkf45", "rk4"])
    if kind == "lines":
        return dict(kind=kind, n=_log_int(rng, 1, 20000), method=method, tol=tol,
                    precision=rng.choice(["fp32c", "fp32c", "mixed", "fp64"]), **_box(rng, 48, 256))
    if kind == "map":
        return dict(kind=kind, nu=_log_int(rng, 32, 768), nv=_log_int(rng, 32, 768), method=method, tol=tol,
                    precision=rng.choice(["fp32c", "fp32c", "mixed", "fp64"]), **_box(rng, 48, 256))
    if kind == "plane":
        return dict(kind=kind, nu=_log_int(rng, 64, 1000), nv=_log_int(rng, 64, 1000), method=method, tol=tol,
                    precision="fp32c", **_box(rng, 64, 320))
    if kind == "cube":
        return dict(kind=kind, sx=_log_int(rng, 24, 400), sy=_log_int(rng, 24, 120), sz=_log_int(rng, 24, 120),
                    method="rkf45", tol=tol, precision="fp32c", nx=_log_int(rng, 128, 512),
                    ny=_log_int(rng, 96, 256), nz=_log_int(rng, 96, 256))
    if kind == "batch":
        return dict(kind=kind, requests=rng.randint(2, 12), side_lo=_log_int(rng, 16, 64),
                    side_hi=_log_int(rng, 128, 600), precision="fp32c", **_box(rng, 64, 256))
    if kind == "neighbour":
        return dict(kind=kind, nu=_log_int(rng, 64, 1000), nv=_log_int(rng, 64, 1000), method=method,
                    precision=rng.choice(["fp32c", "fp32c", "fp32c", "fp64"]), **_box(rng, 64, 256))
    if kind == "stretch":
        return dict(kind=kind, nu=_log_int(rng, 64, 1000), nv=_log_int(rng, 64, 1000),
                    precision=rng.choice(["fp32c", "fp32c", "fp64"]), **_box(rng, 64, 256))
    if kind == "twist":
        return dict(kind=kind, nu=_log_int(rng, 64, 512), nv=_log_int(rng, 64, 512), tol=tol, precision="fp32c",
                    **_box(rng, 64, 256))
    if kind == "dropin":
        return dict(kind=kind, nu=_log_int(rng, 48, 384), nv=_log_int(rng, 48, 384),
                    tracer=rng.choice(["scott", "rkf45", "rk4"]), **_box(rng, 64, 256))
    return dict(kind=kind, nu=_log_int(rng, 64, 256), nv=_log_int(rng, 64, 256), tol=tol, precision="fp32c",
                **_box(rng, 64, 320))


# ------------------------------------------------------------------ inputs
def _shape(case):
    return int(case["nx"]), int(case["ny"]), int(case["nz"])


def _field(shape, seed, dtype=torch.float32, axes=None, rope=False):
    """Random sub-surface point sources (x, y over the box, depth 0.05..0.3,
    normal charges) at the nodes of [-1, 1]^2 x [0, 2], or at the node
    coordinates ``axes`` (in units of a tenth of theirs); three (nx, ny, nz)
    tensors, x fastest in memory."""
    rng = np.random.default_rng(seed)
    count = 8 if rope else 40
    px, py = rng.uniform(-1.0, 1.0, count), rng.uniform(-1.0, 1.0, count)
    depth, q = rng.uniform(0.05, 0.3, count), rng.normal(0.0, 0.3 if rope else 1.0, count)
    if axes is None:
        half = 2.0 if rope else 1.0
        spans = ((-half, half), (-1.0, 1.0), (0.0, 2.0))
        ax = [torch.linspace(lo, hi, n, dtype=torch.float64, device=DEV) for n, (lo, hi) in zip(shape, spans)]
    else:
        ax = [torch.as_tensor(np.asarray(a, np.float64) / 10.0, device=DEV) for a in axes]
    x, y, z = ax[0].view(1, 1, -1), ax[1].view(1, -1, 1), ax[2].view(-1, 1, 1)
    b = [torch.zeros((shape[2], shape[1], shape[0]), dtype=torch.float64, device=DEV) for _ in range(3)]
    for i in range(count):
        dx, dy, dz = x - (2.0 if rope else 1.0) * px[i], y - py[i], z + depth[i]
        r2 = dx * dx + dy * dy + dz * dz
        w = q[i] * r2.rsqrt() / r2
        b[0] += w * dx
        b[1] += w * dy
        b[2] += w * dz
    if rope:  # a uniform-twist rope along x, one and a half turns, radius 0.2 at height 0.4
        t = 2.0 * math.pi * 1.5 / 4.0
        ry, rz = y, z - 0.4
        r2 = ry * ry + rz * rz
        s = (r2 <= 0.04).to(torch.float64) / (1.0 + t * t * r2)
        b[0] += s
        b[1] += -t * rz * s
        b[2] += t * ry * s
    return [c.to(dtype).permute(2, 1, 0) for c in b]


def _grid_z(case, seed, z=0.0):
    """Seeds of a constant-z map over the whole box, rows = y; (n, 3)."""
    nx, ny, _ = _shape(case)
    j = np.random.default_rng(seed + 77).uniform(0.0, 0.1, 4)
    x = torch.linspace(float(j[0]), nx - 1 - float(j[1]), case["nu"], device=DEV)
    y = torch.linspace(float(j[2]), ny - 1 - float(j[3]), case["nv"], device=DEV)
    yy, xx = torch.meshgrid(y, x, indexing="ij")
    return torch.stack([xx.reshape(-1), yy.reshape(-1), torch.full_like(xx, z).reshape(-1)], 1).contiguous()


def _line_seeds(case, seed):
    nx, ny, nz = _shape(case)
    rng = np.random.default_rng(seed + 78)
    p = rng.uniform(0.05, 0.95, (case["n"], 3)) * np.array([nx - 1, ny - 1, 0.3 * (nz - 1)])
    p = torch.as_tensor(p.astype(np.float32), device=DEV)
    return [p[:, i].contiguous() for i in range(3)]


def _abc(case, seed):
    """A vertical-ish cut from the lower boundary up through the box."""
    nx, ny, nz = _shape(case)
    j = np.random.default_rng(seed + 79).uniform(0.0, 0.1, 6)
    hi = np.array([nx - 1, ny - 1, nz - 1], float)
    a = (0.05 + j[:3] * [1, 1, 0]) * hi * [1, 1, 0]
    b = np.array([0.9 + j[3], 0.75 + j[4], 0.0]) * hi
    return a, b, a + np.array([0.0, 0.05 + j[5], 0.6]) * hi


def _batch_requests(case, seed):
    shapes = [_shape(case), (64, 64, 64), (case["ny"], case["nz"], case["nx"])]
    fields = [fq.Field(*_field(s, seed + 11 * i)) for i, s in enumerate(shapes)]
    rng = np.random.default_rng(seed + 80)
    reqs = []
    for k in range(case["requests"]):
        f = k % 3
        hi = np.array(shapes[f], float) - 1
        a, b, c = (rng.uniform(0, 1, 3) * hi for _ in range(3))
        # sides from the smallest to the largest in equal ratios, so that every seed is the same work
        t = k / max(1, case["requests"] - 1)
        side = int(round(case["side_lo"] ** (1 - t) * case["side_hi"] ** t))
        x, y, z = fq.synth.plane_seeds_abc_torch(a, b, c, side, side, device=DEV)
        reqs.append(dict(field=fields[f], x=x, y=y, z=z, method="rk4" if k % 2 else "rkf45",
                         tol=10.0 ** rng.uniform(-7.0, -5.0), step=0.25))
    return reqs


def _dropin_args(case, seed):
    """The arrays a notebook allocates before it calls the kernel."""
    b = [c.permute(2, 1, 0).contiguous().reshape(-1) for c in _field(_shape(case), seed)]
    s = _grid_z(case, seed, z=0.0 if case["tracer"] == "scott" else 1e-4)
    n = s.shape[0]
    one = lambda v, dt: torch.tensor([v], dtype=dt, device=DEV)  # noqa: E731
    dummy = torch.zeros((1, 1), dtype=torch.float32, device=DEV)
    f32 = lambda k: [torch.zeros(n, dtype=torch.float32, device=DEV) for _ in range(k)]  # noqa: E731
    flag = lambda: torch.zeros(n, dtype=torch.int32, device=DEV)  # noqa: E731
    out = {}
    args = b + [torch.tensor(_shape(case), dtype=torch.int32, device=DEV), dummy, dummy, dummy, dummy,
                torch.tensor([False], device=DEV), *(s[:, i].contiguous() for i in range(3)),
                torch.tensor([0.0, 0.0, 1.0], device=DEV)]
    names = ["start_x", "start_y", "start_z", "flag_start", "end_x", "end_y", "end_z", "flag_end", "b_x", "b_y", "b_z"]
    names += ["q_0", "q_perp"] if case["tracer"] == "scott" else ["b_flag", "bs_x", "bs_y", "bs_z", "be_x", "be_y", "be_z"]
    for k in names:
        out[k] = flag() if "flag" in k else f32(1)[0]
        args.append(out[k])
    out["line_len"] = torch.zeros(n, dtype=torch.float64, device=DEV)
    tol = math.sqrt(10.0) / 1000 if case["tracer"] == "scott" else 0.5
    args += [one(0.125, torch.float32), one(n, torch.int64), out["line_len"], one(tol, torch.float32)]
    return tuple(args), out


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind == "lines":
        st["seeds"] = _line_seeds(case, seed)
        st["field"] = fq.Field(*_field(_shape(case), seed))
    elif kind == "map":
        dtype = torch.float64 if case["precision"] == "fp64" else torch.float32
        st["seeds"] = _grid_z(case, seed)
        st["field"] = fq.Field(*_field(_shape(case), seed, dtype))
    elif kind == "plane":
        st["abc"] = _abc(case, seed)
        st["field"] = fq.Field(*_field(_shape(case), seed))
    elif kind == "cube":
        j = np.random.default_rng(seed + 81).uniform(0.0, 0.1, 3)
        st["axes"] = [torch.linspace(float(j[i]), n - 1.1 + float(j[i]), case[k], device=DEV)
                      for i, (k, n) in enumerate(zip(("sx", "sy", "sz"), _shape(case)))]
        st["field"] = fq.Field(*_field(_shape(case), seed, rope=True))
    elif kind == "batch":
        st["batch"] = ScottBatch(_batch_requests(case, seed), precision=case["precision"])
    elif kind == "neighbour":
        st["seeds"] = _grid_z(case, seed, z=1e-4)
        st["stride"] = (case["nx"] - 1) / (case["nu"] - 1)
        st["field"] = fq.Field(*_field(_shape(case), seed))
    elif kind == "stretch":
        spans = ((-10.0, 10.0), (-10.0, 10.0), (0.0, 20.0))
        axes = [fq.synth.stretched_axis(n, lo, hi, k, s) for n, (lo, hi), k, s in
                zip(_shape(case), spans, ("sinh", "sinh", "geometric"), (1.5, 1.5, 3.0))]
        j = np.random.default_rng(seed + 82).uniform(0.0, 0.05, 2)
        x = torch.linspace(-9.5 + float(j[0]), 9.5, case["nu"], device=DEV)
        y = torch.linspace(-9.5 + float(j[1]), 9.5, case["nv"], device=DEV)
        yy, xx = torch.meshgrid(y, x, indexing="ij")
        st["seeds"] = [xx.reshape(-1).contiguous(), yy.reshape(-1).contiguous(),
                       torch.full_like(xx, 1e-3).reshape(-1)]
        st["field"] = fq.Field(*_field(_shape(case), seed, axes=axes), axes=axes, lookup="bisect")
    elif kind == "twist":
        b = _field(_shape(case), seed)
        s = _grid_z(case, seed)
        st["seeds"] = [s[:, i].contiguous() for i in range(3)]
        st["field"] = fq.Field(*b, current=postproc.curl_index(*b))
    elif kind == "dropin":
        st["args"], st["out"] = _dropin_args(case, seed)
        st["kernel"] = {"scott": fq.kernels.compileTraceBlineScott, "rkf45": fq.kernels.compileTraceBlineAdaptive,
                        "rk4": fq.kernels.compileTraceBlineRK4}[case["tracer"]]()
    elif kind == "snapshot":
        st["b"] = _field(_shape(case), seed)
        st["seeds"] = _grid_z(case, seed)
    else:
        raise ValueError(kind)
    return st


# --------------------------------------------------------------------- run
def _arrays(r):
    return {k: v for k, v in r.items() if isinstance(v, torch.Tensor)}


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "lines":
        return _arrays(fq.trace_scott(st["field"], *st["seeds"], method=case["method"], step=0.25,
                                      tol=case["tol"] or 1e-6, precision=case["precision"]))
    if kind == "map":
        return qmap.scott_qmap(st["field"], st["seeds"], (case["nv"], case["nu"]), method=case["method"],
                               tol=case["tol"] or 1e-6, precision=case["precision"])
    if kind == "plane":
        return qmap.scott_qmap_plane(st["field"], ("abc", *st["abc"]), case["nu"], case["nv"], method=case["method"],
                                     tol=case["tol"], precision=case["precision"])
    if kind == "cube":
        return qmap.scott_qcube(st["field"], *st["axes"], method=case["method"], tol=case["tol"],
                                precision=case["precision"])
    if kind == "batch":
        st["batch"].run()
        return st["batch"].results
    if kind == "neighbour":
        r = qmap.neighbour_qmap(st["field"], st["seeds"], (case["nv"], case["nu"]), st["stride"],
                                method=case["method"], step=0.125, tol_coef=0.5, pseudo_tol_scale=0.2,
                                precision=case["precision"])
        return dict(q_all=r["q_all"], n_pseudo=r["n_pseudo"], traces=r["traces"])
    if kind == "stretch":
        return _arrays(fq.trace_plain(st["field"], *st["seeds"], method="rkf45", step=0.01, tol_coef=1e-2,
                                      precision=case["precision"], schedule="per_line", outputs=PLAIN_OUTPUTS))
    if kind == "twist":
        return _arrays(fq.trace_scott(st["field"], *st["seeds"], tol=case["tol"], precision=case["precision"],
                                      outputs=SCOTT_OUTPUTS + ("twist",)))
    if kind == "dropin":
        st["kernel"]((28, 1), (128, 1, 1), st["args"])
        return st["out"]
    with fq.Field(*st["b"]) as field:
        return qmap.scott_qmap(field, st["seeds"], (case["nv"], case["nu"]), tol=case["tol"],
                               precision=case["precision"])


# -------------------------------------------------------------------- work
# Right-hand-side evaluations of a line: fixed steps go by the line's length,
# adaptive ones by the curvature it meets; per line and per cell of the box's
# mean side, as the tracers count them on these fields.
def _evals(case):
    side = (case["nx"] + case["ny"] + case["nz"]) / 3.0
    per_cell = {"lines": 3.0, "map": 3.0, "plane": 3.0, "cube": 5.0, "batch": 4.0, "neighbour": 0.5, "stretch": 0.8,
                "twist": 3.0, "dropin": 3.0, "snapshot": 3.0}[case["kind"]]
    if case.get("method") == "rk4" or case.get("tracer") == "rk4":
        per_cell = 10.0
    elif case.get("tracer") == "rkf45":
        per_cell = 0.5
    return side * per_cell


def _lines(case):
    kind = case["kind"]
    if kind == "lines":
        return case["n"]
    if kind == "cube":
        return case["sx"] * case["sy"] * case["sz"]
    if kind == "batch":
        m = case["requests"]
        return sum((case["side_lo"] ** (1 - k / max(1, m - 1)) * case["side_hi"] ** (k / max(1, m - 1))) ** 2
                   for k in range(m))
    return case["nu"] * case["nv"]


def work(case):
    """Field nodes and seeds read once, outputs written once; the flops of the
    right-hand sides (three trilinear values and their gradient, the
    normalisation, two directional derivatives; a value alone for the plain
    tracers)."""
    kind = case["kind"]
    n = _lines(case)
    node = 24 if case.get("precision") == "fp64" else 12
    cells = case["nx"] * case["ny"] * case["nz"]
    plain = kind in ("neighbour", "stretch") or case.get("tracer") in ("rkf45", "rk4")
    out = {"cube": 20, "batch": 20}.get(kind, 84 if plain else 68)
    if kind == "twist":
        node, out = 2 * node, out + 8
    return {"bytes": float(cells * node + n * (12 + out)), "flops": float(n * _evals(case) * (90 if plain else 350))}


# ------------------------------------------------------------------- exact
class _Lines64:
    """The Scott tracer of plain grid-index boxes in 64 bits: B trilinear with
    the position clamped to the box, the 9-vector (x, u, v) with
    du/ds = (u.grad) b, grad b the central quotient of b over +-1e-3 cells;
    Fehlberg 4(5) with the position error against an absolute tolerance, or
    RK4; each side ends where it leaves the box, on the linear crossing of the
    step with the face (far faces at index N)."""

    A = ((), (1 / 4,), (3 / 32, 9 / 32), (1932 / 2197, -7200 / 2197, 7296 / 2197),
         (439 / 216, -8.0, 3680 / 513, -845 / 4104), (-8 / 27, 2.0, -3544 / 2565, 1859 / 4104, -11 / 40))
    B5 = (16 / 135, 0.0, 6656 / 12825, 28561 / 56430, -9 / 50, 2 / 55)
    ERR = (1 / 360, 0.0, -128 / 4275, -2197 / 75240, 1 / 50, 2 / 55)

    def __init__(self, comps, method, step, tol):
        self.n = torch.tensor(comps[0].shape, dtype=torch.float64, device=DEV)
        self.dims = tuple(comps[0].shape)
        self.flat = torch.stack([c.permute(2, 1, 0).reshape(-1).double() for c in comps], 1)
        self.method, self.step, self.tol = method, step, tol

    def raw(self, p):
        nx, ny, nz = self.dims
        q = torch.minimum(p.clamp(min=0.0), self.n - 1)
        c = torch.minimum(q.floor(), self.n - 2)
        w = (q - c).unsqueeze(-1)
        i = c.long()
        base = (i[..., 2] * ny + i[..., 1]) * nx + i[..., 0]
        v = [self.flat[base + o] for o in (0, 1, nx, nx + 1, nx * ny, nx * ny + 1, nx * ny + nx, nx * ny + nx + 1)]
        v = [v[k] + w[..., 0, :] * (v[k + 1] - v[k]) for k in (0, 2, 4, 6)]
        v = [v[k] + w[..., 1, :] * (v[k + 1] - v[k]) for k in (0, 2)]
        return v[0] + w[..., 2, :] * (v[1] - v[0])

    def unit(self, p):
        b = self.raw(p)
        return b / b.norm(dim=-1, keepdim=True)

    def rhs(self, y):
        h = 1e-3 * torch.eye(3, dtype=torch.float64, device=DEV)
        x = y[:, 0]
        p = torch.cat([x.unsqueeze(1), x.unsqueeze(1) + h, x.unsqueeze(1) - h], 1)
        b = self.unit(p)
        grad = (b[:, 1:4] - b[:, 4:7]) / 2e-3
        return torch.cat([b[:, :1], y[:, 1:] @ grad], 1)

    def attempt(self, y, s):
        s = s.view(-1, 1, 1)
        if self.method == "rk4":
            k1 = s * self.rhs(y)
            k2 = s * self.rhs(y + 0.5 * k1)
            k3 = s * self.rhs(y + 0.5 * k2)
            return (k1 + 2 * k2 + 2 * k3 + s * self.rhs(y + k3)) / 6, None
        k = []
        for row in self.A:
            k.append(s * self.rhs(y + sum(a * kk for a, kk in zip(row, k)) if row else y))
        return (sum(b * kk for b, kk in zip(self.B5, k) if b),
                sum(e * kk[:, 0] for e, kk in zip(self.ERR, k) if e).norm(dim=1))

    def classes(self, p):
        m = self.n - 1
        x, y, z = p.unbind(1)
        lo, hi = p < 0, p >= m
        below = p < m
        inside = (x >= 0) & (y > 0) & (z >= 0) & (p <= m).all(1)
        fl = torch.full_like(x, 42, dtype=torch.long)
        for a in range(3):
            o = [d for d in range(3) if d != a]
            fl = torch.where(lo[:, a] & ~lo[:, o[0]] & ~lo[:, o[1]] & below.all(1), 2 * a + 1, fl)
            fl = torch.where(~lo.any(1) & hi[:, a] & below[:, o[0]] & below[:, o[1]], 2 * a + 2, fl)
        return torch.where(inside, 0, fl)

    def side(self, y, s, length, steps, d, live):
        """One direction of the lines `live`; footpoints as (n, 3, 3) with their class (-42: the line stops)."""
        foot, flag = y.clone(), torch.zeros(len(y), dtype=torch.long, device=DEV)
        lim = 2.0 * float(sum(self.dims))
        on = torch.nonzero(live & (length < lim) & (steps < 10000)).reshape(-1)
        y = y.clone()
        while on.numel():
            inc, err = self.attempt(y[on], s[on] * d)
            ok = torch.ones(on.numel(), dtype=torch.bool, device=DEV)
            if err is not None:
                scale = (self.tol / err / 11.09) ** 0.2
                ok = scale >= 0.618
                s[on] = torch.where(ok, (s[on] * scale).clamp(0.1, 100.0), s[on] * 0.618)
            a, inc, now = y[on][ok], inc[ok], on[ok]
            new = a + inc
            dl = inc[:, 0].norm(dim=1)
            fl = self.classes(new[:, 0])
            out = fl > 0
            length[now] += torch.where(out, torch.zeros_like(dl), dl)
            steps[now] += 1
            y[now] = torch.where(out.view(-1, 1, 1), a, new)
            foot[now] = y[now]
            flag[now] = torch.where(fl == 42, -42, 0)
            face = out & (fl <= 6)
            if bool(face.any()):
                fa, fb, ff, fi = a[face], new[face], fl[face], now[face]
                dim = (ff - 1) // 2
                pick = lambda t: t.gather(1, dim.view(-1, 1)).squeeze(1)  # noqa: E731
                pm = torch.where(ff % 2 == 1, 0.0, self.n[dim])
                p1, p2 = pick(fa[:, 0]), pick(fb[:, 0])
                wa = ((p2 - pm) / (p2 - p1)).view(-1, 1, 1)
                foot[fi] = fa * wa + fb * (1 - wa)
                length[fi] += (pm - p1).abs() / (1e-4 + pick(self.unit(fa[:, 0])).abs())
                flag[fi] = ff
            stop = torch.zeros(len(y), dtype=torch.bool, device=DEV)
            stop[now] = out
            on = on[~stop[on] & (length[on] < lim) & (steps[on] < 10000)]
        return foot, flag

    def trace(self, x, y, z):
        p0 = torch.stack([x, y, z], 1).double()
        n = len(p0)
        b = self.raw(p0)
        b0 = b / b.norm(dim=1, keepdim=True)
        v0 = torch.stack([b0[:, 1], -b0[:, 0], torch.zeros_like(b0[:, 0])], 1)
        v0 = v0 - (v0 * b0).sum(1, keepdim=True) * b0
        v0 = v0 / v0.norm(dim=1, keepdim=True)
        u0 = torch.linalg.cross(b0, v0)
        y0 = torch.stack([p0, u0 / u0.norm(dim=1, keepdim=True), v0], 1)
        s = torch.full((n,), self.step, dtype=torch.float64, device=DEV)
        length, steps = torch.zeros_like(s), torch.zeros(n, dtype=torch.long, device=DEV)
        ends, gone = [], torch.zeros(n, dtype=torch.bool, device=DEV)
        for d in (-1, 1):
            short = (p0[:, 2] < 1e-6) & (b0[:, 2] * d < 0)  # the seed itself is on the lower face
            foot, flag = self.side(y0, s, length, steps, d, ~short & ~gone)
            flag = torch.where(short & ~gone, 5, flag)
            gone = gone | (flag == -42)
            ends.append((foot, flag))
        (fs, cs), (fe, ce) = ends
        seed = torch.minimum(p0.clamp(min=1e-4), self.n - 1 - 1e-4)
        bt = self.raw(seed)
        q0, qp = self.q(fs, cs, fe, ce, b.norm(dim=1))
        r = dict(start=fs[:, 0], end=fe[:, 0], b_this=bt)
        r = {"%s_%s" % (k, c): t[:, i] for k, t in r.items() for i, c in enumerate("xyz")}
        return dict(r, line_len=length, q_0=torch.where(gone, 0.0, q0), q_perp=torch.where(gone, 0.0, qp))

    def q(self, fs, cs, fe, ce, nb):
        bs, be = self.raw(fs[:, 0]), self.raw(fe[:, 0])
        ok = (cs >= 1) & (cs <= 6) & (ce >= 1) & (ce <= 6)
        axis = lambda c: ((c.clamp(1, 6) - 1) // 2).view(-1, 1)  # noqa: E731
        out = []
        for flat in (True, False):
            proj, norm = [], []
            for f, c, bb in ((fs, cs, bs), (fe, ce, be)):
                if flat:  # onto the face along B
                    bn = bb.gather(1, axis(c))
                    w = f[:, 1:].gather(2, axis(c).view(-1, 1, 1).expand(-1, 2, 1)) / bn.unsqueeze(1)
                    proj.append(f[:, 1:] - w * bb.unsqueeze(1))
                else:     # onto the plane across B
                    bn = bb.norm(dim=1, keepdim=True)
                    bu = (bb / bn).unsqueeze(1)
                    proj.append(f[:, 1:] - (f[:, 1:] * bu).sum(2, keepdim=True) * bu)
                norm.append(bn.squeeze(1))
            (us, vs), (ue, ve) = (p.unbind(1) for p in proj)
            dot = lambda p, q: (p * q).sum(1)  # noqa: E731
            num = dot(ue, ue) * dot(vs, vs) + dot(us, us) * dot(ve, ve) - 2 * dot(ue, ve) * dot(us, vs)
            q = num.abs() / (nb * nb / (norm[0] * norm[1])).abs()
            out.append(torch.where(ok, q, torch.nan))
        return out


def exact(case, seed):
    """64-bit values of the traces of small Scott maps.  Adaptive steps are
    steered by an error estimate that round-off forks on some lines, and the
    largest Q of a map are of lines that amplify it without bound, so Q has a
    value of its own only where the step is fixed and the whole path is 64
    bits.  The z of the start points is zero but for the round-off of the
    landing and a few lines at the box's edge, where such a fork decides
    which face they reach.  The longer jobs would take minutes here."""
    kind = case["kind"]
    if kind not in ("lines", "map", "snapshot", "twist") or _lines(case) > 300000:
        return None
    if case.get("method") == "rk4" and case["precision"] != "fp64" and _lines(case) > 70000:
        return None
    dtype = torch.float64 if kind == "map" and case["precision"] == "fp64" else torch.float32
    lines = _Lines64(_field(_shape(case), seed, dtype), case.get("method", "rkf45"), 0.25, case["tol"] or 1e-6)
    if kind == "lines":
        shape, s = (case["n"],), _line_seeds(case, seed)
    else:
        g = _grid_z(case, seed)
        shape, s = (case["nv"], case["nu"]) if kind != "twist" else (len(g),), [g[:, i] for i in range(3)]
    r = {k: v.reshape(shape) for k, v in lines.trace(*s).items()}
    r.update({k: None for k in ("flag_start", "flag_end", "evals", "start_z")})
    if case.get("method") != "rk4" or case["precision"] != "fp64":
        r.update(q_0=None, q_perp=None)
    if kind == "twist":
        r["twist"] = None
    return r
