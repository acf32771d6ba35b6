"""fp32 plans whose axes are transformed by sums (no axis above 128 cells, at
most 2^24 products): lengths of one mode, odd, prime, the longest, both sides
of the limits, either mode order, both signs, strided modes and batches,
against the same algorithm in FP64."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("modes", [(1, 1), (1, 64), (64, 3), (17, 33), (64, 64), (65, 20),
                                   (1, 1, 1), (2, 31, 9), (24, 20, 16), (33, 31, 29), (35, 34, 33)])
@pytest.mark.parametrize("order,sign,upsampfac", [("cmcl", -1, 2.0), ("fft", 1, 1.25)])
def test_small_axes(modes, order, sign, upsampfac):
    import torch

    import neonufft_amd as nnf
    rng = np.random.default_rng(31)
    tol, m, n = 1e-4, 700, int(np.prod(modes))
    x = [rng.uniform(-np.pi, np.pi, m).astype(np.float32) for _ in modes]
    c = (rng.standard_normal(m) + 1j * rng.standard_normal(m)).astype(np.complex64)
    f = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)
    opt = nnf.Options(tol=tol, upsampfac=upsampfac,
                      order=nnf.ModeOrder.FFT if order == "fft" else nnf.ModeOrder.CMCL)
    plan = nnf.Plan(opt, sign, m, [torch.from_numpy(v).cuda() for v in x], modes)
    # modes strided by two along x: only every other entry may be touched
    st = [2 * int(np.prod(modes[:d])) for d in range(len(modes))]
    wide = torch.full((2 * n,), 7.0, dtype=torch.complex64, device="cuda")
    plan.transform_type_1(torch.from_numpy(c).cuda(), wide, st)
    win = torch.zeros(2 * n, dtype=torch.complex64, device="cuda")
    win[::2] = torch.from_numpy(f).cuda()
    back = torch.zeros(m, dtype=torch.complex64, device="cuda")
    plan.transform_type_2(win, st, back)
    torch.cuda.synchronize()
    assert bool((wide[1::2] == 7.0).all())
    x64 = [v.astype(np.float64) for v in x]
    shape = modes[::-1]
    ours, fin = wide[::2].cpu().numpy().reshape(shape), f.reshape(shape)
    if order == "fft":  # the oracle's arrays are in CMCL order
        ours, fin = np.fft.fftshift(ours), np.fft.fftshift(fin)
    # the fp32 share of every parity test: 3e-6 + 0.04 tol, of the sums' rms
    # size (rounding scales with the strengths; one or two sums may cancel)
    bound = 3e-6 + 0.04 * tol
    ref1 = O.nufft1(x64, c.astype(np.complex128), modes, sign, tol, upsampfac)
    size = max(np.linalg.norm(ref1), np.sqrt(n) * np.linalg.norm(c))
    assert np.linalg.norm(ours.ravel() - ref1.ravel()) < bound * size
    ref2 = O.nufft2(x64, fin.ravel().astype(np.complex128), modes, sign, tol, upsampfac)
    assert O.rel_l2(back.cpu().numpy(), ref2) < bound
