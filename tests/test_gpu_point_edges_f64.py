"""fp64 points a hair to either side of whole and half cells, around the edges
of bins and of the period, at the rounding bound.

An even kernel jumps on whole cells, where the last bit of a folded coordinate
decides about a weight of exp(-beta); 1e-9 cell beside them it does not (a
folded coordinate is off by about n 2^-52 < 1e-13 cells), and the weight there,
which grows with the square root of the distance, is off by less than 1e-13.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import neonufft_amd as nnf
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,modes", [(1, (600,)), (2, (70, 45)), (2, (64, 128)), (3, (40, 24, 21))])
@pytest.mark.parametrize("tol", [1e-4, 1e-5, 1e-6, 1e-7, 1e-9])  # ns 5, 6, 7, 8, 10
def test_edges(dim, modes, tol):
    rng = np.random.default_rng(5)
    m, xs = 4000, []
    for d in range(dim):
        n = 2 * modes[d]
        base = rng.choice(np.concatenate([np.arange(0, n), [n]]), m)
        xi = base + rng.choice([1e-9, -1e-9, 0.5 + 1e-9, 0.5 - 1e-9, 1e-3, -1e-3, 0.25], m)
        xs.append(xi / n * 2 * np.pi - np.pi)
    c = rng.standard_normal(m) + 1j * rng.standard_normal(m)
    nm = int(np.prod(modes))
    f = rng.standard_normal(nm) + 1j * rng.standard_normal(nm)
    plan = nnf.Plan(nnf.Options(tol=tol), -1, m, [torch.from_numpy(x).cuda() for x in xs], modes)
    out = torch.zeros(nm, dtype=torch.complex128, device="cuda")
    plan.transform_type_1(torch.from_numpy(c).cuda(), out)
    back = torch.zeros(m, dtype=torch.complex128, device="cuda")
    plan.transform_type_2(torch.from_numpy(f).cuda(), None, back)
    torch.cuda.synchronize()
    assert O.rel_l2(out.cpu().numpy(), O.nufft1(xs, c, modes, -1, tol)) < 1e-10
    assert O.rel_l2(back.cpu().numpy(), O.nufft2(xs, f, modes, -1, tol)) < 1e-10
