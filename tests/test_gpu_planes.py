"""The 3D fp64 plane kernels (tiles of at most 16 x 16 cells, points ordered by
first plane) against the same algorithm in FP64 (oracle).

Sizes: kernel widths at both ends of the range the kernels take, grids whose
last bins are partial, bins of one point, chunks of exactly 128 points and one
more, subproblems that split (one dense bin), and point sets whose planes are
mostly empty.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _points(kind, m, rng):
    if kind == "uniform":
        return [rng.uniform(-np.pi, np.pi, m) for _ in range(3)]
    if kind == "cell":  # one bin holds everything: chunks and split subproblems
        return [rng.uniform(0.3, 0.34, m) for _ in range(3)]
    # two far planes: long runs of empty planes between them
    x = [rng.uniform(-np.pi, np.pi, m) for _ in range(2)]
    return x + [np.where(rng.random(m) < 0.5, 0.5, 1.9) + rng.uniform(0, 1e-3, m)]


@pytest.mark.parametrize("tol", [1e-1, 1e-4, 1e-8, 1e-9, 1e-11])  # ns 2, 5, 9, 10, 12
@pytest.mark.parametrize("kind,m,modes", [
    ("uniform", 1, (6, 5, 7)), ("uniform", 3000, (30, 21, 40)), ("uniform", 40000, (17, 24, 19)),
    ("cell", 128, (24, 20, 16)), ("cell", 129, (24, 20, 16)), ("cell", 5000, (24, 20, 16)),
    ("planes", 700, (20, 20, 64))])
def test_plane_kernels(tol, kind, m, modes):
    import torch

    import neonufft_amd as nnf
    rng = np.random.default_rng(11)
    x = _points(kind, m, rng)
    c = rng.standard_normal(m) + 1j * rng.standard_normal(m)
    n = int(np.prod(modes))
    f = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    dev = [torch.from_numpy(v).cuda() for v in x]
    plan = nnf.Plan(nnf.Options(tol=tol), -1, m, dev, modes)
    out = torch.zeros(n, dtype=torch.complex128, device="cuda")
    plan.transform_type_1(torch.from_numpy(c).cuda(), out)
    back = torch.zeros(m, dtype=torch.complex128, device="cuda")
    plan.transform_type_2(torch.from_numpy(f).cuda(), None, back)
    torch.cuda.synchronize()
    # the same sums in another order: rounding of at most a few thousand terms
    # per cell, the bound of every fp64 parity test
    assert O.rel_l2(out.cpu().numpy(), O.nufft1(x, c, modes, -1, tol)) < 1e-10
    assert O.rel_l2(back.cpu().numpy(), O.nufft2(x, f, modes, -1, tol)) < 1e-10


@pytest.mark.parametrize("counts", [(500, 1, 4000)])
def test_plane_batch(counts):
    import torch

    import neonufft_amd as nnf
    rng = np.random.default_rng(12)
    tol, modes = 1e-7, [(20, 16, 18), (9, 12, 7), (24, 24, 24)]
    xs = [[rng.uniform(-np.pi, np.pi, m) for _ in range(3)] for m in counts]
    dev = [[torch.from_numpy(v).cuda() for v in x] for x in xs]
    plan = nnf.BatchPlan(nnf.Options(tol=tol), -1, list(counts), dev, modes)
    cs = [rng.standard_normal(m) + 1j * rng.standard_normal(m) for m in counts]
    outs = [torch.zeros(int(np.prod(n)), dtype=torch.complex128, device="cuda") for n in modes]
    plan.transform_type_1([torch.from_numpy(c).cuda() for c in cs], outs)
    back = [torch.zeros(m, dtype=torch.complex128, device="cuda") for m in counts]
    plan.transform_type_2(outs, back)
    torch.cuda.synchronize()
    for x, c, n, o, b in zip(xs, cs, modes, outs, back):
        ref = O.nufft1(x, c, n, -1, tol)
        assert O.rel_l2(o.cpu().numpy(), ref) < 1e-10
        assert O.rel_l2(b.cpu().numpy(), O.nufft2(x, o.cpu().numpy(), n, -1, tol)) < 1e-10
