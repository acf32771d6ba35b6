"""Host-side sizing rules, compiled from params.cpp on the CPU: the bin edges
that a plan reports give the same bins when they are passed back, and the fp64
kernel polynomials meet their stated error."""
import os
import random
import shutil
import subprocess

import numpy as np
import pytest

from neonufft_amd import build as B

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include "params.hpp"
#include <cstdio>
#include <cstring>
// lines: "bins dim n0 n1 n2 ns elem_bytes b0 b1 b2 planes" or "pairs ns beta"
int main() {
  char what[16];
  while (std::scanf("%15s", what) == 1) {
    if (!std::strcmp(what, "bins")) {
      int dim, ns, elem, planes, b[3];
      long long n[3];
      if (std::scanf("%d %lld %lld %lld %d %d %d %d %d %d", &dim, n, n + 1, n + 2, &ns, &elem, b,
                     b + 1, b + 2, &planes) != 10)
        return 1;
      const nnf::IntType nn[3] = {n[0], n[1], n[2]};
      const nnf::BinGeom g = nnf::choose_bins(dim, nn, ns, elem, b, planes != 0);
      std::printf("%d %d %d\n", g.bin[0], g.bin[1], g.bin[2]);
    } else {
      int ns;
      double beta;
      if (std::scanf("%d %lf", &ns, &beta) != 2) return 1;
      double c[8 * (nnf::kPairDegree + 1)] = {};
      nnf::fit_pairs(ns, beta, c);
      for (double v : c) std::printf("%a ", v);
      std::printf("\n");
    }
  }
}
"""


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    if not os.path.exists(B.HOSTCXX) and shutil.which(B.HOSTCXX) is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("params")
    src, exe = d / "driver.cpp", d / "driver"
    src.write_text(DRIVER)
    r = subprocess.run([B.HOSTCXX, "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__",
                        f"-I{os.path.join(ROOT, 'include')}", "-I/opt/rocm/include", f"-I{B.CSRC}",
                        str(src), os.path.join(B.CSRC, "params.cpp"), "-o", str(exe),
                        "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(lines):
        r = subprocess.run([str(exe)], input="\n".join(lines) + "\n", capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        return r.stdout.splitlines()

    return run


def test_reported_bins_round_trip(ask):
    rng = random.Random(3)
    shapes = [(3, (192, 150, 160), 9, 16, 1), (3, (192, 150, 160), 9, 16, 0)]
    for _ in range(6000):
        dim = rng.choice((1, 2, 3, 3, 3))
        top = {1: 500000, 2: 3000, 3: 600}[dim]
        ns = rng.randint(2, 16)
        n = [max(2 * ns, int(np.exp(rng.uniform(np.log(4), np.log(top))))) for _ in range(dim)]
        shapes.append((dim, tuple(n), ns, rng.choice((8, 16)), rng.randint(0, 1)))
    fmt = lambda d, n, ns, e, b, p: "bins %d %s %d %d %s %d" % (
        d, " ".join(map(str, list(n) + [1] * (3 - d))), ns, e, " ".join(map(str, b)), p)
    first = ask([fmt(d, n, ns, e, (0, 0, 0), p) for d, n, ns, e, p in shapes])
    edges = [tuple(map(int, l.split())) for l in first]
    # back as plans are made from them: unused axes 0, whatever the density
    for planes in (0, 1):
        again = ask([fmt(d, n, ns, e, b[:d] + (0,) * (3 - d), planes)
                     for (d, n, ns, e, _), b in zip(shapes, edges)])
        for s, b, l in zip(shapes, edges, again):
            assert tuple(map(int, l.split())) == b, (s, b, l)
    assert edges[0] == (8, 8, 24)  # (was widened to 8 x 10 x 24, out of the plane kernels)


def test_pair_polynomials(ask):
    """Against the kernel in extended precision: within 1.8e-15 over the widths
    and shape parameters that plans use, 2.5e-16 of rounding in the sum allowed."""
    X = np.longdouble
    cases = [(ns, f * ns) for ns in range(3, 17) for f in (1.5, 2.3, 3.05)]
    got = ask(["pairs %d %r" % c for c in cases])
    x = (np.arange(4001, dtype=X)) / 4000
    y = 2 * x - 1
    for (ns, beta), line in zip(cases, got):
        c = np.array([float.fromhex(v) for v in line.split()]).reshape(8, 17)
        for j in range(1, (ns + 1) // 2):
            t = x + j - X(ns) / 2
            want = np.exp(X(beta) * (np.sqrt(1 - 4 * t * t / (X(ns) * ns)) - 1))
            v = np.zeros_like(x)
            for k in range(16, -1, -1):
                v = v * y + X(c[j, k])
            assert float(np.max(np.abs(v - want))) < 1.8e-15 + 2.5e-16, (ns, beta, j)
