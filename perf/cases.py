"""The transforms whose speed this repository tracks, as a user's program calls them.

Kinds of a case:
  type1 / type2   a plan whose points are set, one transform per pass (an iterative solver, many
                  right-hand sides of one point set)
  points_type1    the points change with every pass: set_points, then type 1 (particles that move,
                  a trajectory per frame)
  type3           add_input, transform, reset of a type-3 plan: sources to targets, both off-grid
  batch           many independent 2D type-1 transforms of uneven sizes through one BatchPlan
                  (visibility sets per channel)

Points are uniform in [-pi, pi)^d, or a mixture of 16 Gaussians ("clustered"); strengths and modes
are complex standard normals. Mode arrays are contiguous with x fastest, in either mode order.
"""
import math

import torch

import neonufft_amd as nnf

PI = math.pi


def _case(name, kind, dtype, points, modes, tol, order="cmcl", upsampfac=2.0, layout="uniform",
          **more):
    c = {"kind": kind, "dtype": dtype, "points": points, "dim": len(modes), "tol": tol,
         "order": order, "upsampfac": upsampfac, "layout": layout}
    if name:
        c["name"] = name
    for d, m in enumerate(modes):
        c["n%d" % d] = m
    c.update(more)
    return c


def listed():
    return [
        # the smallest calls: a few thousand points, where launches and latency are all there is
        _case("small_2d_type1", "type1", "f32", 2000, (50, 40), 1e-3),
        _case("small_3d_type2", "type2", "f32", 4000, (24, 20, 16), 1e-5),
        # one long line: 1D spectra of irregularly sampled series
        _case("line_1d_type1", "type1", "f32", 1000000, (200000,), 1e-6),
        # double precision at a tight tolerance, one image: 2D, 1e-9
        _case("image_2d_type1_f64", "type1", "f64", 100000, (256, 256), 1e-9),
        # new points on every call, an image of ragged size (a grid that is no power of two)
        _case("points_2d_type1", "points_type1", "f32", 1000000, (500, 450), 1e-4),
        # the volume of the benchmark, both directions: 1e7 points, 128^3 modes, 1e-5
        _case("volume_3d_type1", "type1", "f32", 10000000, (128, 128, 128), 1e-5),
        _case("volume_3d_type2", "type2", "f32", 10000000, (128, 128, 128), 1e-5),
        # clustered points on a large volume at a tighter tolerance: 2e7 points, 256^3 modes
        _case("clustered_3d_type2", "type2", "f32", 20000000, (256, 256, 256), 1e-6,
              layout="clustered"),
        # a volume of ragged size in FFT order, single precision
        _case("ragged_3d_type2", "type2", "f32", 2000000, (100, 90, 81), 1e-4, order="fft"),
        # a volume of ragged size, double precision
        _case("ragged_3d_type1_f64", "type1", "f64", 1000000, (96, 75, 80), 1e-8),
        # flat, baseline-like sources of large magnitude to off-grid targets, double precision
        _case("offgrid_3d_type3_f64", "type3", "f64", 2000000, (1, 1, 1), 1e-6, targets=1000000,
              x0=1e4, x1=1e4, x2=50.0, s0=0.02, s1=0.02, s2=1.0),
        # 256 uneven images in one call
        _case("batch_2d_type1", "batch", "f32", 1000000, (1024, 1024), 1e-5, count=256,
              least=10000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _modes(rng, dim, most):
    """Modes per axis of one size class, every other volume ragged."""
    edge = _log_int(rng, *((1000, most) if dim == 1 else (16, most)))
    if rng.random() < 0.4:  # a power of two, equal on all axes
        return (1 << max(4, int(round(math.log2(edge)))),) * dim
    return tuple(max(8, int(edge * rng.uniform(0.7, 1.0))) for _ in range(dim))


def draw(rng):
    kind = rng.choice(("type1", "type2", "type1", "type2", "points_type1", "type3", "batch"))
    if kind == "batch":
        return _case(None, "batch", "f32", _log_int(rng, 30000, 600000), (512, 512),
                     rng.choice((1e-4, 1e-5)), order=rng.choice(("cmcl", "fft")),
                     count=_log_int(rng, 8, 128), least=_log_int(rng, 1000, 20000))
    dtype = rng.choice(("f32", "f32", "f64"))
    dim = rng.choice((1, 2, 2, 3, 3, 3))
    tol = rng.choice((1e-3, 1e-4, 1e-5, 1e-6) if dtype == "f32" else (1e-6, 1e-8, 1e-9, 1e-10))
    if kind == "type3":
        dim = rng.choice((2, 3))
        most = 1000000 if dtype == "f32" else 300000
        more = {"targets": _log_int(rng, 1000, most)}
        for d in range(dim):
            x = math.exp(rng.uniform(math.log(3.0), math.log(1e4)))
            more["x%d" % d] = round(x, 3)
            more["s%d" % d] = round(rng.uniform(10.0, 120.0 if dim == 3 else 400.0) / x, 6)
        return _case(None, kind, dtype, _log_int(rng, 1000, most), (1,) * dim, tol, **more)
    most = {1: 4000000, 2: 4000000, 3: 6000000 if dtype == "f32" else 1000000}[dim]
    modes = _modes(rng, dim, {1: 500000, 2: 1000, 3: 128 if dtype == "f32" else 90}[dim])
    return _case(None, kind, dtype, _log_int(rng, 1000, most), modes, tol,
                 order=rng.choice(("cmcl", "cmcl", "fft")),
                 upsampfac=rng.choice((2.0, 2.0, 2.0, 2.0, 1.25))
                 if tol >= (1e-4 if dtype == "f32" else 1e-6) else 2.0,
                 layout=rng.choice(("uniform", "uniform", "uniform", "clustered")))


# ---- inputs ---------------------------------------------------------------

def _modes_of(case):
    return [int(case["n%d" % d]) for d in range(case["dim"])]


def _real(case):
    return torch.float32 if case["dtype"] == "f32" else torch.float64


def _complex(case):
    return torch.complex64 if case["dtype"] == "f32" else torch.complex128


def _normal(n, dtype, g):
    return torch.randn(n, dtype=dtype, device="cuda", generator=g)


def _points(case, m, g):
    if case["layout"] == "uniform":
        return [((torch.rand(m, dtype=torch.float64, device="cuda", generator=g) * 2 - 1) * PI)
                .to(_real(case)) for _ in range(case["dim"])]
    which = torch.randint(16, (m,), device="cuda", generator=g)
    loc = []
    for _ in range(case["dim"]):
        centre = (torch.rand(16, dtype=torch.float64, device="cuda", generator=g) * 2 - 1) * PI
        v = centre[which] + 0.05 * torch.randn(m, dtype=torch.float64, device="cuda", generator=g)
        loc.append((torch.remainder(v + PI, 2 * PI) - PI).to(_real(case)))
    return loc


def _box(case, prefix, m, g):
    return [((torch.rand(m, dtype=torch.float64, device="cuda", generator=g) * 2 - 1)
             * case["%s%d" % (prefix, d)]).to(_real(case)) for d in range(case["dim"])]


def _options(case):
    return nnf.Options(tol=case["tol"], upsampfac=case["upsampfac"],
                       order=nnf.ModeOrder.FFT if case["order"] == "fft" else nnf.ModeOrder.CMCL)


def _batch_sizes(case):
    """Point counts spread over [least, points] in their logarithm; edges n0, n0 / 2, n0 / 4."""
    n, lo, hi = case["count"], math.log(case["least"]), math.log(case["points"])
    counts = [int(math.exp(lo + (i + 0.5) / n * (hi - lo))) for i in range(n)]
    return counts, [(case["n0"] >> (i % 3), case["n1"] >> (i % 3)) for i in range(n)]


def _inputs(case, seed):
    """Everything the exact sums need: coordinates, strengths or modes, targets."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    cdt, kind = _complex(case), case["kind"]
    if kind == "batch":
        counts, modes = _batch_sizes(case)
        loc = [_points(case, m, g) for m in counts]
        return {"counts": counts, "modes": modes, "loc": loc,
                "c": [_normal(m, cdt, g) for m in counts]}
    m = case["points"]
    if kind == "type3":
        return {"loc": _box(case, "x", m, g), "target": _box(case, "s", case["targets"], g),
                "c": _normal(m, cdt, g)}
    loc = _points(case, m, g)
    return {"loc": loc, "c": _normal(math.prod(_modes_of(case)) if kind == "type2" else m, cdt, g)}


def prepare(case, seed):
    s = _inputs(case, seed)
    opt, kind, cdt = _options(case), case["kind"], _complex(case)
    s["kind"] = kind
    if kind == "batch":
        s["plan"] = nnf.BatchPlan(opt, -1, s["counts"], s["loc"], s["modes"], use_graph=True)
        sizes = [math.prod(m) for m in s["modes"]]
        s["out"] = torch.zeros(sum(sizes), dtype=cdt, device="cuda")
        s["outs"] = list(torch.split(s["out"], sizes))
    elif kind == "type3":
        s["plan"] = nnf.PlanT3(opt, -1, case["points"], s["loc"], case["targets"], s["target"])
        s["out"] = torch.zeros(case["targets"], dtype=cdt, device="cuda")
    else:
        sign = 1 if kind == "type2" else -1
        modes = _modes_of(case)
        s["plan"] = nnf.Plan(opt, sign, case["points"], s["loc"], modes)
        n = case["points"] if kind == "type2" else math.prod(modes)
        s["out"] = torch.zeros(n, dtype=cdt, device="cuda")
        s["points"] = case["points"]
    return s


def run(state):
    plan, kind = state["plan"], state["kind"]
    if kind == "batch":
        plan.transform_type_1(state["c"], state["outs"])
    elif kind == "type3":
        plan.add_input(state["c"])
        plan.transform(state["out"])
        plan.reset()
    elif kind == "type2":
        plan.transform_type_2(state["c"], None, state["out"])
    else:
        if kind == "points_type1":
            plan.set_points(state["points"], state["loc"])
        plan.transform_type_1(state["c"], state["out"])
    return state["out"]


# ---- the least work -------------------------------------------------------

def _width(tol, upsampfac):
    """Kernel width the tolerance asks for."""
    if upsampfac == 2.0:
        ns = math.ceil(-math.log10(tol / 10.0))
    else:
        ns = math.ceil(-math.log(tol) / (PI * math.sqrt(1.0 - 1.0 / upsampfac)))
    return max(2, min(16, ns))


def _transform_work(case, m, cells, modes, targets=0):
    real = 4 if case["dtype"] == "f32" else 8
    per = _width(case["tol"], case["upsampfac"]) ** case["dim"]
    points = m + targets
    return (points * (case["dim"] + 2) * real + modes * 2 * real,
            4.0 * points * per + 5.0 * cells * math.log2(max(2.0, cells)))


def work(case):
    sigma, dim = case["upsampfac"], case["dim"]
    if case["kind"] == "batch":
        each = [_transform_work(case, m, math.prod(n) * sigma ** dim, math.prod(n))
                for m, n in zip(*_batch_sizes(case))]
        return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}
    if case["kind"] == "type3":
        ns = _width(case["tol"], sigma)
        spread = math.prod(2 * sigma * case["x%d" % d] * case["s%d" % d] / PI + ns + 1
                           for d in range(dim))
        b, f = _transform_work(case, case["points"], spread * sigma ** dim, 0, case["targets"])
    else:
        n = math.prod(_modes_of(case))
        b, f = _transform_work(case, case["points"], n * sigma ** dim, n)
    return {"bytes": b, "flops": f}


# ---- the sums in 64 bits --------------------------------------------------

def _wave(n, order, x, sign):
    """exp(sign i k x) for the n modes of one axis, [n, points]."""
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    k = torch.where(k < n - n // 2, k, k - n) if order == "fft" else k - n // 2
    a = sign * k[:, None] * x[None, :]
    return torch.complex(torch.cos(a), torch.sin(a))


def _sum_type1(loc, c, modes, order, sign):
    """Direct sum of one transform by matrix products over chunks of points, x fastest."""
    rest = math.prod(modes[1:])
    out = torch.zeros(rest, modes[0], dtype=torch.complex128, device="cuda")
    chunk = max(64, min(c.numel(), int(1.2e8 / max(rest, modes[0]))))
    for i in range(0, c.numel(), chunk):
        x = [v[i:i + chunk].double() for v in loc]
        right = _wave(modes[0], order, x[0], sign) * c[i:i + chunk].to(torch.complex128)
        left = torch.ones(1, x[0].numel(), dtype=torch.complex128, device="cuda")
        for d in range(1, len(modes)):
            e = _wave(modes[d], order, x[d], sign)
            left = (e[:, None, :] * left[None, :, :]).reshape(-1, x[0].numel())
        out += left @ right.T
    return out.reshape(-1)


def _sum_type2(loc, f, modes, order, sign):
    rest, m = math.prod(modes[1:]), loc[0].numel()
    grid = f.to(torch.complex128).reshape(rest, modes[0])
    out = torch.empty(m, dtype=torch.complex128, device="cuda")
    chunk = max(64, min(m, int(1.2e8 / max(rest, modes[0]))))
    for i in range(0, m, chunk):
        x = [v[i:i + chunk].double() for v in loc]
        left = torch.ones(1, x[0].numel(), dtype=torch.complex128, device="cuda")
        for d in range(1, len(modes)):
            e = _wave(modes[d], order, x[d], sign)
            left = (e[:, None, :] * left[None, :, :]).reshape(-1, x[0].numel())
        out[i:i + chunk] = ((grid.T @ left) * _wave(modes[0], order, x[0], sign)).sum(0)
    return out


def _sum_type3(loc, c, target, sign):
    x = torch.stack([v.double() for v in loc], 1)
    s = torch.stack([v.double() for v in target], 1)
    c = c.to(torch.complex128)
    out = torch.empty(s.shape[0], dtype=torch.complex128, device="cuda")
    chunk = max(1, int(1.2e8 / x.shape[0]))
    for j in range(0, s.shape[0], chunk):
        a = sign * (s[j:j + chunk] @ x.T)
        out[j:j + chunk] = torch.complex(torch.cos(a), torch.sin(a)) @ c
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        pairs = float(sum(m * math.prod(n) for m, n in zip(*_batch_sizes(case))))
    elif kind == "type3":
        pairs = 25.0 * case["points"] * case["targets"]
    else:
        pairs = (25.0 if case["dim"] == 1 else 1.0) * case["points"] * math.prod(_modes_of(case))
    if pairs > 3e13:  # over about 20 seconds
        return None
    s = _inputs(case, seed)
    if kind == "batch":
        return torch.cat([_sum_type1(l, c, m, case["order"], -1)
                          for l, c, m in zip(s["loc"], s["c"], s["modes"])])
    if kind == "type3":
        return _sum_type3(s["loc"], s["c"], s["target"], -1)
    if kind == "type2":
        return _sum_type2(s["loc"], s["c"], _modes_of(case), case["order"], 1)
    return _sum_type1(s["loc"], s["c"], _modes_of(case), case["order"], -1)
