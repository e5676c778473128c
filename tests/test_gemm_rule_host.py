"""Which kernel a product runs on (alfq_gemm_rule.h, compiled here by itself): the sizes that the GPU
tests use to reach a kernel, so that a change of the rule cannot move them to another one unseen."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DIRECT, TILE_64, TILE_32, LDS_16_32, LDS_16 = range(5)

MAIN = """
#include <cstdio>
#include "alfq_gemm_rule.h"
int main() {
  int m, n, k, b, policy, tile;
  while (std::scanf("%d %d %d %d %d %d", &m, &n, &k, &b, &policy, &tile) == 6)
    std::printf("%d\\n", (int)gemm_kernel_for(m, n, k, b, policy, tile != 0));
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "alf_amd", "csrc"),
                    str(d / "main.cpp"), "-o", str(d / "rule")], check=True)

    def ask(m, n, k, b=1, policy=0, tile=1):
        r = subprocess.run([str(d / "rule")], input=f"{m} {n} {k} {b} {policy} {tile}\n", capture_output=True, text=True,
                           check=True)
        return int(r.stdout)
    return ask


@pytest.mark.parametrize("k", [1, 15, 16, 17, 33, 47])
def test_sizes_of_the_tile_tests(rule, k):
    assert rule(1473, 1500, k) == TILE_64
    assert rule(507, 510, k) == TILE_32
    assert rule(507, 510, k, policy=3) == DIRECT


@pytest.mark.parametrize("n,b", [(99, 32), (125, 128), (63, 512)])
def test_sizes_of_the_batches(rule, n, b):
    assert rule(n, n, n, b) == (TILE_32 if n == 99 else TILE_64)
    assert rule(n, n, n, 1) == DIRECT
    assert rule(n, n, n, b, policy=2) != TILE_64
    assert rule(n, n, n, b, tile=0) != TILE_64
