"""A refused set_output_points leaves a type-3 plan as it was: its points and
the bins they were sorted into belong together, whichever bins the refused
count would have asked for."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import neonufft_amd as nnf

from test_gpu_plan import CDT, RDT, cplx, dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("held,refused", [(4000, 3), (40, 400000)])
def test_refused_output_points(prec, held, refused):
    rng = np.random.default_rng(8)
    tol, m = 1e-6, 500
    x = [rng.uniform(-9.0, 9.0, m) for _ in range(3)]
    s = [rng.uniform(-1.2, 1.2, held) for _ in range(3)]
    c = cplx(rng, m, prec)
    plan = nnf.PlanT3(nnf.Options(tol=tol), -1, m, [dev(v, RDT[prec]) for v in x], held,
                      [dev(v, RDT[prec]) for v in s])
    out, again = (torch.zeros(held, dtype=CDT[prec], device="cuda") for _ in range(2))
    plan.add_input(dev(c, CDT[prec]))
    plan.transform(out)
    with pytest.raises(nnf.InputError):
        plan.set_output_points(refused, [0, 0, 0])  # null coordinates
    plan.transform(again)
    torch.cuda.synchronize()
    assert np.array_equal(again.cpu().numpy(), out.cpu().numpy())
    a = np.outer(s[0], x[0]) + np.outer(s[1], x[1]) + np.outer(s[2], x[2])
    ref = np.exp(-1j * a) @ c.astype(np.complex128)
    got = again.cpu().numpy()
    # fp32 coordinates: phases of up to 33 rad rounded to 2^-24 of each factor
    bound = 2e-5 if prec == "f32" else 10 * tol
    assert np.linalg.norm(got - ref) < bound * np.linalg.norm(ref)
