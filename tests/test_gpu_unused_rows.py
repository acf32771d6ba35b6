"""Grids most of whose rows no point's kernel meets: the row kernels leave
those rows out (type 2) or write zero modes for them (type 1).

Points crowd around the period's ends, a bin edge, or one cell, so the rows in
use wrap around the grid and end inside pencils. The grid must be whole again
where a caller can see it: interpolation of other points, accumulation, and
the grid itself.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [((32, 32, 32), 1e-5), ((16, 64, 32), 1e-3), ((64, 25, 21), 1e-4), ((128, 100), 1e-5),
         ((64, 64), 1e-3)]


def _points(dim, m, at, rng):
    return [np.mod(at + rng.uniform(-0.05, 0.05, m) + np.pi, 2 * np.pi) - np.pi for _ in range(dim)]


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("modes,tol", CASES)
@pytest.mark.parametrize("at", [np.pi, 0.0, 1.3])
def test_unused_rows(prec, modes, tol, at):
    import torch

    import neonufft_amd as nnf
    rdt, cdt = (np.float32, np.complex64) if prec == "f32" else (np.float64, np.complex128)
    rng = np.random.default_rng(21)
    dim, m, n = len(modes), 600, int(np.prod(modes))
    x = [v.astype(rdt) for v in _points(dim, m, at, rng)]
    y = [rng.uniform(-np.pi, np.pi, m).astype(rdt) for _ in range(dim)]
    c = (rng.standard_normal(m) + 1j * rng.standard_normal(m)).astype(cdt)
    f = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(cdt)
    cu = lambda v: torch.from_numpy(v).cuda()
    dx, dy, dc, df = [cu(v) for v in x], [cu(v) for v in y], cu(c), cu(f)
    plan = nnf.Plan(nnf.Options(tol=tol), -1, m, dx, modes)
    # garbage of another transform in the grid and the intermediates first
    plan.set_points(m, dy)
    other, back, t1 = torch.zeros_like(dc), torch.zeros_like(dc), torch.zeros_like(df)
    plan.transform_type_2(df * 3, None, other)
    plan.transform_type_1(dc, t1)
    plan.set_points(m, dx)
    plan.transform_type_2(df, None, back)
    plan.set_points(m, dy)
    plan.interp(other)  # the rows left out are needed here
    plan.set_points(m, dx)
    plan.transform_type_1(dc, t1)
    torch.cuda.synchronize()
    # fp32 share of the parity bound: 3e-6 + 0.04 tol; fp64: rounding, 1e-10,
    # or the kernel's jump at a last bit (1e-10 holds: no point on a cell)
    bound = 3e-6 + 0.04 * tol if prec == "f32" else 1e-10
    up = lambda a: a.astype(np.complex128)
    x64, y64 = [v.astype(np.float64) for v in x], [v.astype(np.float64) for v in y]
    assert O.rel_l2(back.cpu().numpy(), O.nufft2(x64, up(f), modes, -1, tol)) < bound
    assert O.rel_l2(other.cpu().numpy(), O.nufft2(y64, up(f), modes, -1, tol)) < bound
    assert O.rel_l2(t1.cpu().numpy(), O.nufft1(x64, up(c), modes, -1, tol)) < bound
