"""The choice between the row-adaptive tiles and the others (csrc/rows_rule.h) where both were measured, and at the limits of
what it looks at."""
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
  long long v, a, b, c, d, e;
  while (std::scanf("%lld %lld %lld %lld %lld %lld", &v, &a, &b, &c, &d, &e) == 6)
    std::printf("%d\\n", v < 0 ? gmoe::rows_one_launch_pays(a, b, c, d, e) : gmoe::rows_pays((gmoe::RowsKind)v, a, b, c, d, e));
}
"""
NN, GLU, NT, GLU_BWD = range(4)
# kind, experts, rows per expert, K, M, us on the other tiles and on the row-adaptive ones
MEASURED = [
    (GLU, 8, 382, 4096, 28672, 975.7, 649.6), (GLU, 64, 139, 2048, 2816, 258.8, 165.3),
    (GLU, 16, 640, 1024, 5632, 188.6, 138.3), (GLU, 2, 668, 3936, 6400, 105.5, 79.09),
    (GLU, 4, 608, 3232, 1024, 39.14, 55.32), (NN, 8, 382, 14336, 4096, 437.4, 336.5),
    (NN, 64, 139, 1408, 2048, 120, 89.89), (NN, 16, 640, 2816, 1024, 81.26, 62.77),
    (NN, 32, 1024, 2048, 7168, 1165, 808.8), (NN, 64, 267, 576, 832, 44.72, 36.03),
    (NN, 64, 921, 1536, 128, 52.02, 58.89), (NN, 24, 1832, 640, 4480, 380.2, 284.4),
    (NN, 4, 336, 4832, 2432, 53.2, 72.43), (NT, 8, 382, 28672, 4096, 860.3, 628.4),
    (NT, 16, 640, 5632, 1024, 159.3, 116.2), (NT, 1, 1111, 2048, 11264, 68.47, 53.81),
    (NT, 1, 1111, 5632, 2048, 49.44, 77.36), (NT, 8, 740, 14336, 4096, 636.2, 530),
    (NT, 64, 1000, 640, 128, 27.89, 30.87), (NT, 8, 1000, 28672, 4096, 1439, 1413),
    (NT, 8, 600, 2056, 4104, 115.9, 112), (GLU_BWD, 8, 382, 4096, 14336, 469.8, 381.9),
    (GLU_BWD, 16, 640, 1024, 2816, 102.7, 110.8), (GLU_BWD, 8, 1000, 4096, 14336, 1138, 835.9),
    (GLU_BWD, 48, 192, 1024, 1024, 48.16, 47.56), (GLU_BWD, 32, 1024, 7168, 2048, 1119, 834.7),
    (NN, 8, 363, 512, 5120, 32.26, 31.75), (NN, 24, 137, 2560, 10240, 414.5, 268),
    (NN, 24, 5374, 2688, 224, 246, 174.1), (NN, 32, 941, 768, 128, 17.59, 24.39),
    (NN, 2, 656, 1280, 1280, 14.29, 23.23), (NN, 4, 1701, 10848, 160, 79.07, 132.5),
    (GLU, 32, 208, 128, 512, 12.15, 13.35), (GLU, 64, 389, 512, 14336, 908.1, 621.9),
    (GLU, 4, 1318, 1952, 1504, 60.4, 49.96), (GLU, 4, 103, 768, 1024, 12.61, 18.11),
    (GLU, 8, 121, 7168, 256, 64.92, 94.84), (NT, 1, 1185, 1792, 7552, 45.63, 42.35),
    (NT, 4, 938, 12544, 2112, 282.8, 216.3), (NT, 32, 203, 1392, 1968, 76.45, 59.1),
    (NT, 24, 222, 12256, 192, 81.63, 193.8), (NT, 4, 1769, 1408, 512, 16.43, 23.71),
    (NT, 1, 866, 19968, 1536, 95.51, 260.5), (GLU_BWD, 60, 386, 6272, 2688, 1231, 909.3),
    (GLU_BWD, 24, 124, 128, 2560, 20.62, 22.03), (GLU_BWD, 2, 1917, 1888, 3936, 96.82, 75.48),
    (GLU_BWD, 6, 599, 304, 544, 15.36, 29.33), (GLU_BWD, 4, 322, 4992, 1024, 52.84, 73.34),
]


@pytest.fixture(scope="module")
def evaluate(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    folder = tmp_path_factory.mktemp("rule")
    (folder / "rule.cpp").write_text(PROGRAM)
    exe = str(folder / "rule")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wno-unknown-pragmas", "-I" + CSRC, str(folder / "rule.cpp"), "-o", exe])

    def run(cases):
        text = "\n".join("%d %d %d %d %d %d" % c for c in cases)
        out = subprocess.run([exe], input=text, text=True, capture_output=True, check=True).stdout.split()
        assert len(out) == len(cases)
        return [int(v) for v in out]

    return run


def test_choice(evaluate):
    """Over the measured launches, short reductions and small launches among them, the choice takes less than 1 % longer than
    the better side of each on average and 15 % at most."""
    got = evaluate([(kind, E, n * E, K, M, 256) for kind, E, n, K, M, _, _ in MEASURED])
    lost = [(c[5], c[6])[v] / min(c[5], c[6]) - 1 for c, v in zip(MEASURED, got)]
    worst = max(zip(lost, MEASURED))
    assert worst[0] < 0.15 and sum(lost) / len(lost) < 0.01, (sum(lost) / len(lost), worst)


def test_few_rows(evaluate):
    """The launch with the activation, from 4 rows per expert on: where its tiles fill nine tenths of their rounds or more.  us in
    the other tiles and in these, as above but with all rows."""
    measured = [(8, 26, 4096, 28672, 319.1, 350.5), (8, 128, 4096, 28672, 331.5, 363.4), (64, 1024, 2048, 2816, 142.1, 131.4),
                (64, 2664, 2048, 2816, 152.3, 139.8), (16, 256, 1024, 5632, 42.6, 46.5), (16, 1024, 1024, 5632, 47, 54.5),
                (32, 8, 7168, 4096, 83.7, 104.9), (4, 128, 128, 512, 8.3, 9.6), (4, 104, 2368, 6400, 30.6, 38.4)]
    got = evaluate([(GLU, *c[:4], 256) for c in measured])
    assert got == [int(c[5] < c[4]) for c in measured]
    assert not any(evaluate([(kind, *c[:4], 256) for c in measured for kind in (NN, NT, GLU_BWD)]))
    # fewer: how many experts have rows is not known
    assert not any(evaluate([(GLU, E, N, 2048, 2816, 256) for E in (1, 8, 64) for N in (1, 2, 3 * E, 4 * E - 1) if N < 4 * E]))


def test_one_launch(evaluate):
    """Short launches of fc1 with its activation are one launch where the host's time decides; longer ones, and none at all, are
    not.  us in one launch and in two."""
    measured = [(4, 128, 128, 512, 9.4, 8.2), (4, 26, 128, 512, 9.2, 8.1), (64, 64, 128, 256, 9.1, 10.9), (8, 128, 512, 1024, 12.5, 10.9),
                (8, 26, 4096, 28672, 350.5, 319.1), (16, 64, 1024, 5632, 45.2, 42.2), (4, 104, 2368, 6400, 38.4, 30.6),
                (6, 132, 1664, 6400, 36, 31)]
    got = evaluate([(-1, *c[:4], 256) for c in measured])
    assert got == [int(c[4] < 15) for c in measured]
    assert not any(evaluate([(-1, E, 0, 128, 512, 256) for E in (1, 64)]))


def test_limits(evaluate):
    """Fewer than 96 rows per expert, with the activation fewer than four: never; one expert and a thousand, the smallest and
    the longest reductions: an answer; the largest launches: always."""
    shapes = [(E, n, K, M) for E in (1, 8, 1024) for n in (0, 1, 95, 96, 2048, 65536) for K in (8, 512, 65536) for M in (8, 4096)]
    large = [(8, 4096, 4096, 28672), (8, 16384, 14336, 4096), (64, 4096, 2048, 2816), (1, 32768, 8192, 8192)]
    for kind in (NN, GLU, NT, GLU_BWD):
        for (E, n, K, M), v in zip(shapes, evaluate([(kind, E, n * E, K, M, 256) for E, n, K, M in shapes])):
            assert v in (0, 1) and not (v and n < (4 if kind == GLU else 96)), (kind, E, n, K, M)
        assert all(evaluate([(kind, E, n * E, K, M, 256) for E, n, K, M in large])), kind
