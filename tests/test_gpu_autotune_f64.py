"""The autotuner over 3D fp64 plans: it can choose the plane tiles, and shapes
that a cache file holds from kernels of another revision are timed again."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import neonufft_amd as nnf

from test_gpu_plan import dev

pytestmark = pytest.mark.gpu


def _points(m):
    rng = np.random.default_rng(9)
    return [dev(rng.uniform(-np.pi, np.pi, m), torch.float64) for _ in range(3)]


@pytest.mark.parametrize("tol,ns", [(1e-8, 9), (1e-10, 11)])
def test_plane_tiles_are_candidates(tol, ns, monkeypatch):
    monkeypatch.setenv("NEONUFFT_AMD_TUNE_CACHE", "")
    nnf._L.lib().nnf_autotune_clear_cache()
    m, modes = 100000, (48, 40, 44)
    x = _points(m)
    opt = nnf.Options(tol=tol)
    t = nnf.autotune(opt, -1, m, x, modes, reps=2)
    assert t["source"] == 0
    # several times faster here than any LDS tile
    assert max(t["bin_size"][:2]) + ns - 1 <= 16, t
    tuned = nnf.Plan(opt, -1, m, x, modes, bin_size="auto").info()
    assert tuned["bin_size"] == t["bin_size"]


def test_shapes_of_another_kernel_revision_are_timed_again(monkeypatch, tmp_path):
    new, old = tmp_path / "new.txt", tmp_path / "old.txt"
    m, modes, opt = 20000, (20, 20, 20), nnf.Options(tol=1e-8)
    x = _points(m)
    clear = nnf._L.lib().nnf_autotune_clear_cache
    monkeypatch.setenv("NEONUFFT_AMD_TUNE_CACHE", str(new))
    clear()
    assert nnf.autotune(opt, -1, m, x, modes, reps=1)["source"] == 0
    line = new.read_text().split(" ")
    # a line as written before revisions were: the library version alone
    old.write_text(" ".join([line[0], nnf.version()] + line[2:]))
    monkeypatch.setenv("NEONUFFT_AMD_TUNE_CACHE", str(old))
    clear()
    assert nnf.autotune(opt, -1, m, x, modes, reps=1)["source"] == 0
    # a line of this revision is read
    same = tmp_path / "same.txt"
    same.write_text(" ".join(line))
    monkeypatch.setenv("NEONUFFT_AMD_TUNE_CACHE", str(same))
    clear()
    assert nnf.autotune(opt, -1, m, x, modes, reps=1)["source"] == 2
