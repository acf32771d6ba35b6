"""Points on and next to the edges of bins and of the period.

A point belongs to the bin of its first kernel cell i0 + floor(ns/2) (mod n);
coordinates whose kernel starts at the last cell of a bin, or wraps past the
end of the grid, are where a wrong bin or relative cell would show.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("dim,modes", [(1, (600,)), (2, (70, 45)), (3, (40, 24, 21))])
@pytest.mark.parametrize("tol", [1e-4, 1e-5])  # odd and even kernel width
def test_edges(prec, dim, modes, tol):
    import torch

    import neonufft_amd as nnf
    rdt, cdt = (np.float32, np.complex64) if prec == "f32" else (np.float64, np.complex128)
    rng = np.random.default_rng(5)
    # cell coordinates at whole and half cells and a hair to either side,
    # around the period's ends and every 8th cell (bin edges are multiples)
    xs = []
    m = 4000
    for d in range(dim):
        n = 2 * modes[d]
        base = rng.choice(np.concatenate([np.arange(0, n, 8), [n - 1, n - 2, n - 3, n]]), m)
        xi = base + rng.choice([0.0, 0.5, -0.5, 1e-3, -1e-3, 0.25], m)
        xs.append((xi / n * 2 * np.pi - np.pi).astype(rdt))
    c = (rng.standard_normal(m) + 1j * rng.standard_normal(m)).astype(cdt)
    f = (rng.standard_normal(modes[::-1]) + 1j * rng.standard_normal(modes[::-1])).astype(cdt).ravel()
    x64 = [x.astype(np.float64) for x in xs]
    dev = [torch.from_numpy(x).cuda() for x in xs]
    plan = nnf.Plan(nnf.Options(tol=tol), -1, m, dev, modes)
    out = torch.zeros(int(np.prod(modes)), dtype=torch.from_numpy(c).dtype, device="cuda")
    plan.transform_type_1(torch.from_numpy(c).cuda(), out)
    back = torch.zeros(m, dtype=out.dtype, device="cuda")
    plan.transform_type_2(torch.from_numpy(f).cuda(), None, back)
    torch.cuda.synchronize()
    # the same algorithm in FP64; fp32 adds its rounding (bound of the fp32
    # share of every parity test: 3e-6 + 0.04 tol)
    bound = 3e-6 + 0.04 * tol if prec == "f32" else 1e-10
    # an even kernel ends on whole cells, where it jumps from exp(-beta) to 0:
    # a point there keeps or loses that weight, per axis, with the last bit of
    # its folded coordinate (beta = 2.3 ns)
    if prec == "f64" and tol == 1e-5:
        bound = dim * np.exp(-2.3 * 6)
    assert O.rel_l2(out.cpu().numpy(), O.nufft1(x64, c.astype(np.complex128), modes, -1, tol)) < bound
    assert O.rel_l2(back.cpu().numpy(), O.nufft2(x64, f.astype(np.complex128), modes, -1, tol)) < bound
