"""Which tiles 3D fp64 plans take: plane tiles (at most 16 x 16 cells in x and y)
at kernel widths 8 to 12, at width 7 below one point in three cells, LDS tiles
otherwise. Both sides of every line, as single plans, batches and
type-3 targets, against the same algorithm in FP64 (direct sums for type 3)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import neonufft_amd as nnf
from oracle import oracle as O

from test_gpu_plan import cplx, dev

pytestmark = pytest.mark.gpu

MODES = (17, 20, 18)
CELLS = 8 * 17 * 20 * 18


def _points(m, rng):
    x = [rng.uniform(-np.pi, np.pi, m) for _ in range(3)]
    return x, [dev(v, torch.float64) for v in x]


@pytest.mark.parametrize("tol,ns,m,planes", [
    (1e-5, 6, 900, False), (1e-6, 7, 900, True), (1e-6, 7, CELLS // 3 - 1, True),
    (1e-6, 7, CELLS // 3 + 1, False), (1e-7, 8, CELLS // 3 + 1, True),
    (1e-11, 12, 900, True), (1e-12, 13, 900, False)])
def test_plan(tol, ns, m, planes):
    rng = np.random.default_rng(m)
    x, dx = _points(m, rng)
    plan = nnf.Plan(nnf.Options(tol=tol), -1, m, dx, MODES)
    info = plan.info()
    assert info["n_spread"] == ns
    assert (max(info["bin_size"][:2]) + ns - 1 <= 16) == planes
    n = int(np.prod(MODES))
    c, f = cplx(rng, m, "f64"), cplx(rng, n, "f64")
    out = torch.zeros(n, dtype=torch.complex128, device="cuda")
    back = torch.zeros(m, dtype=torch.complex128, device="cuda")
    plan.transform_type_1(dev(c, torch.complex128), out)
    plan.transform_type_2(dev(f, torch.complex128), None, back)
    torch.cuda.synchronize()
    # the same sums in another order: the bound of every fp64 parity test
    assert O.rel_l2(out.cpu().numpy(), O.nufft1(x, c, MODES, -1, tol)) < 1e-10
    assert O.rel_l2(back.cpu().numpy(), O.nufft2(x, f, MODES, -1, tol)) < 1e-10


@pytest.mark.parametrize("count", [700, CELLS // 2])
def test_batch(count):
    rng = np.random.default_rng(count)
    tol, modes, counts = 1e-6, [MODES, (20, 20, 20)], [count, count // 7]
    pts = [_points(m, rng) for m in counts]
    plan = nnf.BatchPlan(nnf.Options(tol=tol), -1, counts, [d for _, d in pts], modes)
    cs = [cplx(rng, m, "f64") for m in counts]
    outs = [torch.zeros(int(np.prod(n)), dtype=torch.complex128, device="cuda") for n in modes]
    back = [torch.zeros(m, dtype=torch.complex128, device="cuda") for m in counts]
    plan.transform_type_1([dev(c, torch.complex128) for c in cs], outs)
    plan.transform_type_2(outs, back)
    torch.cuda.synchronize()
    for (x, _), c, n, o, b in zip(pts, cs, modes, outs, back):
        assert O.rel_l2(o.cpu().numpy(), O.nufft1(x, c, n, -1, tol)) < 1e-10
        assert O.rel_l2(b.cpu().numpy(), O.nufft2(x, o.cpu().numpy(), n, -1, tol)) < 1e-10


@pytest.mark.parametrize("tol", [1e-5, 1e-6, 1e-8])
@pytest.mark.parametrize("targets", [60, 6000])
def test_type3(tol, targets):
    rng = np.random.default_rng(targets)
    m = 800
    x = [rng.uniform(-8.0, 8.0, m) for _ in range(3)]
    s = [rng.uniform(-1.1, 1.1, targets) for _ in range(3)]
    c = cplx(rng, m, "f64")
    plan = nnf.PlanT3(nnf.Options(tol=tol), -1, m, [dev(v, torch.float64) for v in x], targets,
                      [dev(v, torch.float64) for v in s])
    out = torch.zeros(targets, dtype=torch.complex128, device="cuda")
    plan.add_input(dev(c, torch.complex128))
    plan.transform(out)
    torch.cuda.synchronize()
    ref = np.exp(-1j * (np.outer(s[0], x[0]) + np.outer(s[1], x[1]) + np.outer(s[2], x[2]))) @ c
    # the kernel's own error: the requested tolerance, per axis and stage
    got = out.cpu().numpy()
    assert np.linalg.norm(got - ref) < 10 * tol * np.linalg.norm(ref)


@pytest.mark.parametrize("prec,tol,modes", [("f64", 1e-8, (96, 75, 80)), ("f64", 1e-6, (31, 64, 29)),
                                            ("f32", 1e-5, (20, 33, 41)), ("f32", 1e-8, (9, 82, 9))])
def test_reported_bins_give_the_same_plan(prec, tol, modes):
    dt = torch.float64 if prec == "f64" else torch.float32
    rng = np.random.default_rng(6)
    dx = [dev(rng.uniform(-np.pi, np.pi, 3000), dt) for _ in range(3)]
    opt = nnf.Options(tol=tol)
    info = nnf.Plan(opt, -1, 3000, dx, modes).info()
    assert nnf.Plan(opt, -1, 3000, dx, modes, bin_size=info["bin_size"]).info() == info


@pytest.mark.parametrize("modes,m", [((12, 12, 12), 40000), ((12, 12, 12), 70), ((40, 40, 40), 30000),
                                     ((64, 64, 64), 30000), ((80, 72, 76), 20000)])
def test_parts_of_subproblems(modes, m):
    """Interpolation cuts subproblems into eight parts (few of them) down to one
    (many); parts of one point, empty ones and full ones."""
    rng = np.random.default_rng(m)
    tol, n = 1e-8, int(np.prod(modes))
    x, dx = _points(m, rng)
    x[0][: m // 2] = rng.uniform(0.2, 0.25, m // 2)  # half of them in few bins
    dx[0] = dev(x[0], torch.float64)
    f = cplx(rng, n, "f64")
    plan = nnf.Plan(nnf.Options(tol=tol), -1, m, dx, modes)
    assert max(plan.info()["bin_size"][:2]) + plan.info()["n_spread"] - 1 <= 16
    back = torch.zeros(m, dtype=torch.complex128, device="cuda")
    plan.transform_type_2(dev(f, torch.complex128), None, back)
    torch.cuda.synchronize()
    assert O.rel_l2(back.cpu().numpy(), O.nufft2(x, f, modes, -1, tol)) < 1e-10
