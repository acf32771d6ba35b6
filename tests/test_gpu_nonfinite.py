"""Interpolation of a grid with infinities and NaN in single cells: a point's
value depends on the cells its kernel meets and on no other, in every
precision and dimension, whichever kernel takes it."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import neonufft_amd as nnf
from oracle import oracle as O

from test_gpu_plan import CDT, RDT, dev, points
from test_gpu_stages import NPC, h2d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tols", [("f32", (1e-1, 1e-5)), ("f64", (1e-1, 1e-4, 1e-8, 1e-11, 1e-13))])
@pytest.mark.parametrize("modes,m", [((12, 10, 11), 700), ((24, 21, 20), 3000), ((30, 25), 900)])
def test_nonfinite_cells_stay_with_their_points(prec, tols, modes, m):
    dim = len(modes)
    for tol in tols:
        rng = np.random.default_rng(17)
        x = points(rng, dim, m, prec)
        plan = nnf.Plan(nnf.Options(tol=tol), -1, m, [dev(v, RDT[prec]) for v in x], modes)
        info = plan.info()
        n, ns, beta = info["grid"], info["n_spread"], info["es_beta"]
        cells = int(np.prod(n))
        grid = rng.standard_normal(cells) + 1j * rng.standard_normal(cells)
        # one component of a cell each, the last cells included
        bad = [np.inf, -np.inf, np.nan]
        for k, cell in enumerate(list(rng.choice(cells, 8, replace=False)) + [0, cells - 1]):
            re, im = grid[cell].real, grid[cell].imag
            grid[cell] = complex(bad[k % 3], im) if k & 1 else complex(re, bad[k % 3])

        def interp(values):
            h2d(plan.fine_grid_ptr(), values.astype(NPC[prec]))
            out = torch.empty(m, dtype=CDT[prec], device="cuda")
            plan.interp(out)
            torch.cuda.synchronize()
            return out.cpu().numpy()

        got = interp(grid)
        finite = lambda v: np.where(np.isfinite(v), v, 0.0)
        zeroed = interp(finite(grid.real) + 1j * finite(grid.imag))
        u = [O.fold(v.astype(np.float64)) for v in x]
        shape = tuple(reversed(n))
        touched = 0
        for part, g in (("real", grid.real), ("imag", grid.imag)):
            ours = getattr(got, part).astype(np.float64)
            fin = getattr(zeroed, part).astype(np.float64)
            # the points that meet a bad cell (weights are positive inside the kernel)
            hit = {}
            for name, at in (("+", np.isposinf(g)), ("-", np.isneginf(g)), ("nan", np.isnan(g))):
                hit[name] = O.interp(n, ns, beta, u, at.astype(np.complex128).reshape(shape)).real != 0
            nan = hit["nan"] | (hit["+"] & hit["-"])
            pos, neg = hit["+"] & ~nan, hit["-"] & ~nan
            clean = ~(nan | pos | neg)
            touched += int((~clean).sum())
            np.testing.assert_array_equal(np.isfinite(ours), clean)
            if prec == "f64":  # (the fp32 fit may go below zero at the kernel's ends)
                np.testing.assert_array_equal(np.isnan(ours), nan)
                np.testing.assert_array_equal(np.isposinf(ours), pos)
                np.testing.assert_array_equal(np.isneginf(ours), neg)
            # the others read the same cells of both grids; their sums may be
            # formed in another order (fp64: at most 16^3 roundings of 2^-53)
            bound = 1e-6 if prec == "f32" else 1e-12
            assert np.linalg.norm(ours[clean] - fin[clean]) < bound * np.linalg.norm(fin)
        assert 0 < touched < 2 * m
