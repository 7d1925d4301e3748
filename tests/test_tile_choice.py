"""Which kernel a product of more than 32 rows takes (csrc/mm_plan.h, host code):
measured times of every kernel at shapes where they differ, and the choice among
them; the workspace covers every plan.  Runs on the CPU."""

from __future__ import annotations

import random
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "metal-marlin_amd" / "csrc"

MAIN = r"""
#include <cstdio>
#include "mm_plan.h"
using namespace mmplan;
// M, N, K, group size, INT4 -> kernel (0 mid-sized, 256, 128 or 64 row tiles) and
// the partial sums' bytes of the mid-sized and the prefill plan
int main() {
  int M, N, K, g, i4;
  while (std::scanf("%d %d %d %d %d", &M, &N, &K, &g, &i4) == 5) {
    const MidPlan m = plan_mid(M, N, K, g, i4);
    const PrefillPlan p = plan_prefill(M, N, K, g, i4);
    const size_t mid = m.wn != 0 && m.ks > 1 ? 4ul * m.ks * cdiv(N, 64 * m.wn) * cdiv(M, 32 * m.rb) *
                                                   (64 * m.wn) * (32 * m.rb) : 0;
    std::printf("%d %zu %zu\n", m.wn != 0 ? 0 : 256 >> p.cfg, mid,
                p.ksplit > 1 ? 4ul * p.ksplit * M * N : 0);
  }
}
"""


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(d / "main.cpp"), "-o",
                    str(d / "plan")], check=True)

    def run(cases):
        text = "".join(f"{m} {n} {k} {g} {int(i4)}\n" for i4, m, n, k, g in cases)
        out = subprocess.run([str(d / "plan")], input=text, capture_output=True, text=True,
                             check=True).stdout
        return [tuple(int(v) for v in line.split()) for line in out.splitlines()]

    return run


# (INT4, M, N, K, group size): us of the mid-sized, the 256-row and the 128-row
# tiles (64-row tiles up to 64 rows), measured on MI355X.  The pair forms are planned
# as one product of 2N columns.
MEASURED = {
    (0, 33, 14336, 4096, 128): (16.1, None, 18.05),
    (0, 48, 8192, 2048, 32): (10.17, None, 16.27),
    (0, 100, 8736, 1664, 32): (11.69, None, 24.46),
    (0, 129, 4096, 4096, 128): (14.96, 86.95, 23.54),
    (0, 200, 512, 4096, 128): (9.34, 86.66, 15.81),
    (0, 640, 14336, 4096, 128): (90.71, 99.0, 116.6),
    (0, 640, 8736, 1664, 32): (30.76, 46.94, 49.65),
    (0, 800, 664, 5376, 128): (17.44, 113.79, 23.97),
    (0, 1024, 4096, 1024, 64): (15.38, 28.01, 28.16),
    (0, 512, 28672, 4096, 128): (138.4, 110.26, 129.36),
    (0, 2048, 6144, 4096, 128): (115.35, 102.36, 122.06),
    (0, 3000, 4096, 14336, 128): (366.87, 332.4, 406.42),
    (0, 6400, 2048, 2048, 128): (74.03, 57.56, 66.28),
    (0, 8192, 4096, 4096, 128): (304.21, 234.5, 266.36),
    (0, 1600, 4096, 1024, 64): (27.49, 29.1, 19.44),
    (0, 1600, 4096, 4096, 128): (71.1, 92.28, 61.7),
    (0, 6400, 1024, 4096, 128): (76.13, 92.01, 64.8),
    (0, 6400, 512, 4096, 128): (45.92, 89.37, 42.22),
    (0, 8192, 856, 3968, 64): (84.23, 89.86, 66.69),
    (1, 64, 4096, 4096, 128): (11.81, None, 19.11),
    (1, 65, 856, 3968, 64): (13.44, None, 27.01),
    (1, 129, 8192, 2048, 32): (20.32, 74.15, 30.87),
    (1, 1024, 4096, 4096, 32): (62.9, 144.9, 71.19),
    (1, 2048, 3072, 1024, 128): (28.5, 35.39, 41.7),
    (1, 33, 6728, 8192, 64): (29.28, None, 23.12),
    (1, 64, 4096, 14336, 64): (28.71, None, 25.43),
    (1, 800, 14336, 4096, 128): (165.06, 128.55, 167.0),
    (1, 1024, 8736, 1664, 64): (70.66, 53.43, 71.94),
    (1, 2500, 28672, 4096, 128): (930.0, 663.11, 805.85),
    (1, 3200, 4096, 4096, 32): (204.31, 147.33, 222.64),
    (1, 100, 14336, 4096, 128): (35.53, None, 31.73),
    (1, 300, 4096, 14336, 128): (111.13, 389.85, 89.22),
    (1, 1600, 4096, 1024, 64): (36.62, 35.68, 25.88),
    (1, 2048, 856, 3968, 64): (45.59, 113.05, 35.17),
    (1, 2500, 664, 5376, 128): (46.82, 151.25, 40.85),
    (1, 4096, 2048, 2048, 32): (72.22, 77.56, 60.83),
}


def test_choice_is_near_the_fastest(choose):
    """Within 8% of the fastest kernel at each of these shapes (the kernels differ by
    8 to 700% there; two boxes by up to 5%)."""
    slow = {}
    for (case, us), (rows, _, _) in zip(MEASURED.items(), choose(MEASURED), strict=True):
        took = us[{0: 0, 256: 1}.get(rows, 2)]
        if took > 1.08 * min(t for t in us if t):
            slow[case] = (rows, us)
    assert not slow


def test_workspace_covers_every_plan(choose):
    """mm_gemm_workspace_bytes knows neither the format nor the group size."""
    import mmfp4
    rng = random.Random(0)
    cases = [(i4, rng.randint(33, 2000), 8 * rng.randint(1, 1024), 128 * rng.randint(1, 112), g)
             for _ in range(400) for g in (32, 64, 128) for i4 in (0, 1)]
    need = mmfp4._lib.load().mm_gemm_workspace_bytes
    head = need(0, 8, 8)          # the counters alone
    for (_, m, n, k, _), (_, mid, prefill) in zip(cases, choose(cases), strict=True):
        assert need(m, n, k) - head >= max(mid, prefill), (m, n, k)
