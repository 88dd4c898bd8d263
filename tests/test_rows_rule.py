"""The choice between the row-adaptive tiles and the others (csrc/rows_rule.h) where both were measured and one is
clearly ahead, and at the limits of what it looks at; and the chunks that the row-adaptive tiles cut rows into."""
import os
import shutil
import subprocess

import pytest

from test_gmm_rows_gpu import EDGES, ROWS

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hetu-galvatron_amd", "csrc")
PROGRAM = """
#define __host__
#define __device__
#include "rows_rule.h"
#include <cstdio>
int main() {
  long long v, a, b, c, d, e;
  while (std::scanf("%lld %lld %lld %lld %lld %lld", &v, &a, &b, &c, &d, &e) == 6) {
    const int units[5] = {(int)a, 0, (int)b, (int)c, (int)d};
    const int col_tiles = (int)(e >> 32);
    std::printf("%d\\n", v < 0 ? gmoe::rows_chunk_units(units, col_tiles, 256, e & 0xffffffff)
                               : gmoe::rows_pays((gmoe::RowsKind)v, a, b, c, d, e));
  }
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
    got = evaluate([(kind, E, n * E, K, M, 256) for kind, E, n, K, M, _, _ in MEASURED])
    wrong = [c for c, v in zip(MEASURED, got) if v != (c[6] < c[5])]
    assert not wrong, wrong
    # no rows, fewer than 96, reductions of up to 512, 2048 rows and more: never; one expert and a thousand: an answer
    shapes = [(E, n, K, M) for E in (1, 8, 1024) for n in (0, 1, 95, 96, 2047, 2048) for K in (8, 512, 520, 4096)
              for M in (8, 128, 4096)]
    for kind in (NN, GLU, NT, GLU_BWD):
        for (E, n, K, M), v in zip(shapes, evaluate([(kind, E, n * E, K, M, 256) for E, n, K, M in shapes])):
            assert v in (0, 1) and not (v and (n < 96 or n >= 2048 or K <= 512)), (kind, E, n, K, M)


def test_chunks(evaluate):
    """Chunks of up to 256, 192 and 128 rows against the rule in Python, for the edge test on the GPU, which reaches all
    three; no rows at all; one tile."""
    def units(rows):
        u = [-(-r // 64) for r in rows]
        return [sum(u)] + [sum(-(-x // size) for x in u) for size in (2, 3, 4)]

    def model(counts, col_tiles, K):
        best, least = 4, None
        for size in (4, 3, 2):
            chunks = counts[size - 1]
            cost = -(-chunks * col_tiles // 256) * (16 + 250 / -(-K // 32) + 4 * counts[0] / max(chunks, 1))
            if least is None or cost < 0.95 * least:
                best, least = size, cost
        return best

    edges = [(units(ROWS * times), cols, K) for K, F, times in EDGES for cols in (-(-F // 128), -(-F // 256))]
    other = [(units(rows), cols, K) for rows in ([0, 0], [1], [640] * 16, [256] * 64, [370] * 8) for cols in (1, 4, 6, 25)
             for K in (520, 1024, 5632)]
    got = evaluate([(-1, *counts, cols << 32 | K) for counts, cols, K in edges + other])
    assert got == [model(*c) for c in edges + other]
    assert set(got[:len(edges)]) == {2, 3, 4}
