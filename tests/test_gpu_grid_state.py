"""The fine grid as the stage calls see it, between transforms, refused calls
and graph replays. Type 2 forms only the rows its points read; whatever reads
the grid afterwards must find all of them.

Points of the first set crowd in one place, so most rows are left out; the
second set is uniform and reads every row.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import neonufft_amd as nnf
from oracle import oracle as O

from test_gpu_stages import d2h

pytestmark = pytest.mark.gpu

TOL = 1e-4
# the fp32 share of every parity test: 3e-6 + 0.04 tol
BOUND = 3e-6 + 0.04 * TOL
SHAPES = [(32, 32, 32), (64, 25, 21), (128, 100)]


class Inputs:
    def __init__(self, modes, seed=41):
        rng = np.random.default_rng(seed)
        self.modes, self.m, self.n = modes, 500, int(np.prod(modes))
        dim, m = len(modes), self.m
        self.x = [rng.uniform(1.2, 1.3, m).astype(np.float32) for _ in range(dim)]
        self.y = [rng.uniform(-np.pi, np.pi, m).astype(np.float32) for _ in range(dim)]
        cplx = lambda k: (rng.standard_normal(k) + 1j * rng.standard_normal(k)).astype(np.complex64)
        self.c, self.f, self.f2 = cplx(m), cplx(self.n), cplx(self.n)
        cu = lambda v: torch.from_numpy(v).cuda()
        self.dx, self.dy = [cu(v) for v in self.x], [cu(v) for v in self.y]
        self.dc, self.df, self.df2 = cu(self.c), cu(self.f), cu(self.f2)

    def plan(self, loc, stream=None):
        return nnf.Plan(nnf.Options(tol=TOL), -1, self.m, loc, self.modes, stream=stream)

    def out(self):
        return torch.zeros(self.m, dtype=torch.complex64, device="cuda")

    def at_y(self, f):
        y = [v.astype(np.float64) for v in self.y]
        return O.nufft2(y, f.astype(np.complex128), self.modes, -1, TOL)

    def whole_grid(self, f):
        """The grid of a plan that forms every row."""
        p = self.plan(self.dx)
        ptr = p.fine_grid_ptr()
        p.transform_type_2(f, None, self.out())
        return d2h(ptr, int(np.prod(p.info()["grid"])), np.complex64)

    def stale(self, p):
        """Another transform's values in every row of the grid."""
        p.set_points(self.m, self.dy)
        p.transform_type_2(self.df2 * 3, None, self.out())
        p.set_points(self.m, self.dx)


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("modes", SHAPES)
def test_refused_type_1_leaves_the_grid(modes):
    v = Inputs(modes)
    p = v.plan(v.dx)
    v.stale(p)
    p.transform_type_2(v.df, None, v.out())
    with pytest.raises(nnf.InputError):
        p.transform_type_1(None, torch.zeros_like(v.df))
    p.set_points(v.m, v.dy)
    out = v.out()
    p.interp(out)
    torch.cuda.synchronize()
    assert rel(out.cpu().numpy(), v.at_y(v.f)) < BOUND


@pytest.mark.parametrize("modes", SHAPES)
def test_accumulating_spread_and_the_grid_after_type_2(modes):
    v = Inputs(modes)
    p = v.plan(v.dx)
    v.stale(p)
    p.transform_type_2(v.df, None, v.out())
    p.spread(v.dc, accumulate=True)
    cells = int(np.prod(p.info()["grid"]))
    got = d2h(p.fine_grid_ptr(), cells, np.complex64)
    ref = v.plan(v.dx)
    ref.spread(v.dc)
    sums = d2h(ref.fine_grid_ptr(), cells, np.complex64)
    want = v.whole_grid(v.df).astype(np.complex128) + sums
    assert rel(got, want) < 1e-6  # the same kernels: one rounding of the sum
    # asked for at once
    p = v.plan(v.dx)
    v.stale(p)
    p.transform_type_2(v.df, None, v.out())
    assert rel(d2h(p.fine_grid_ptr(), cells, np.complex64), v.whole_grid(v.df)) < 1e-6
