"""The choice between the row-adaptive tiles and the others (csrc/rows_rule.h) where both were measured and one is
clearly ahead, and at the limits of what it looks at."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hetu-galvatron_amd", "csrc")
PROGRAM = """
#define __host__
#define __device__
#include "rows_rule.h"
#include <cstdio>
int main() {
  long long kind, E, N, K, M;
  while (std::scanf("%lld %lld %lld %lld %lld", &kind, &E, &N, &K, &M) == 5)
    std::printf("%d\\n", gmoe::rows_pays((gmoe::RowsKind)kind, E, N, K, M, 256));
}
"""
NN, GLU, NT, GLU_BWD = range(4)
# kind, experts, rows per expert, K, M, us on the other tiles and on the row-adaptive ones
MEASURED = [
    (GLU, 8, 382, 4096, 28672, 1004, 724), (GLU, 64, 139, 2048, 2816, 238, 188), (GLU, 16, 640, 1024, 5632, 162, 168),
    (GLU, 2, 668, 3936, 6400, 95, 73), (GLU, 4, 608, 3232, 1024, 33, 46),
    (NN, 8, 382, 14336, 4096, 537, 330), (NN, 64, 139, 1408, 2048, 122, 94), (NN, 16, 640, 2816, 1024, 84, 69),
    (NN, 32, 1024, 2048, 7168, 893, 857), (NN, 64, 267, 576, 832, 34, 41), (NN, 64, 921, 1536, 128, 39, 55),
    (NN, 24, 1832, 640, 4480, 291, 327), (NN, 4, 336, 4832, 2432, 44, 58),
    (NT, 8, 382, 28672, 4096, 1074, 737), (NT, 16, 640, 5632, 1024, 158, 137), (NT, 1, 1111, 2048, 11264, 72, 59),
    (NT, 1, 1111, 5632, 2048, 51, 78), (NT, 8, 740, 14336, 4096, 644, 729), (NT, 64, 1000, 640, 128, 29, 38),
    (NT, 8, 1000, 28672, 4096, 1809, 1891), (NT, 8, 600, 2056, 4104, 120, 156),
    (GLU_BWD, 8, 382, 4096, 14336, 525, 455), (GLU_BWD, 16, 640, 1024, 2816, 128, 119),
    (GLU_BWD, 8, 1000, 4096, 14336, 886, 945), (GLU_BWD, 48, 192, 1024, 1024, 55, 60),
    (GLU_BWD, 32, 1024, 7168, 2048, 911, 1004),
]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_choice(tmp_path):
    (tmp_path / "rule.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "rule")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I" + CSRC, str(tmp_path / "rule.cpp"), "-o", exe])

    def choices(cases):
        text = "\n".join("%d %d %d %d %d" % c for c in cases)
        return [int(v) for v in subprocess.run([exe], input=text, text=True, capture_output=True, check=True).stdout.split()]

    got = choices([(kind, E, n * E, K, M) for kind, E, n, K, M, _, _ in MEASURED])
    wrong = [c for c, v in zip(MEASURED, got) if v != (c[6] < c[5])]
    assert not wrong, wrong
    # no rows, fewer than 96, reductions of up to 512, 2048 rows and more: never; one expert and a thousand: an answer
    shapes = [(E, n, K, M) for E in (1, 8, 1024) for n in (0, 1, 95, 96, 2047, 2048) for K in (8, 512, 520, 4096)
              for M in (8, 128, 4096)]
    for kind in (NN, GLU, NT, GLU_BWD):
        for (E, n, K, M), v in zip(shapes, choices([(kind, E, n * E, K, M) for E, n, K, M in shapes])):
            assert v in (0, 1) and not (v and (n < 96 or n >= 2048 or K <= 512)), (kind, E, n, K, M)
