"""The piece counts of split reductions (csrc/split_rule.h) against the same rule in whole numbers of Python: the
kernels of a 16-bit split launch each come to it for themselves, so a tie may not hang on the rounding of a float."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hetu-galvatron_amd", "csrc")
PROGRAM = """
#define __host__
#define __device__
#include "split_rule.h"
#include <cstdio>
int main() {
  long long a, b, c, d;
  while (std::scanf("%%lld %%lld %%lld %%lld", &a, &b, &c, &d) == 4) std::printf("%%d\\n", gmoe::%s(a, b, c, d));
}
"""


def evaluate(function, cases, tmp_path):
    (tmp_path / "rule.cpp").write_text(PROGRAM % function)
    exe = str(tmp_path / "rule")
    subprocess.check_call(["g++", "-O2", "-I" + CSRC, str(tmp_path / "rule.cpp"), "-o", exe])
    out = subprocess.run([exe], input="\n".join("%d %d %d %d" % c for c in cases), text=True, capture_output=True,
                         check=True).stdout.split()
    assert len(out) == len(cases)
    return [int(v) for v in out]


def model(k_tiles, tiles, slots, stream_ns):
    if tiles == 0:
        return 1
    most = min(slots // tiles, 8, k_tiles)
    if most < 2:
        return 1
    whole, per_piece = 420 * k_tiles, 26 * tiles
    s = max([2] + [n for n in range(2, most + 1) if (2 * n - 1) ** 2 * per_piece <= 4 * whole])
    return s if whole - max(whole // s, stream_ns) > 6000 + per_piece * s else 1


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_pieces(tmp_path):
    cases = [(k, t, slots, ns) for k in (1, 2, 5, 15, 16, 39, 44, 64, 65, 195, 224, 896, 1 << 22)
             for t in (0, 1, 4, 31, 32, 56, 96, 128, 168, 255, 256, 257, 100000) for slots in (2, 511, 512)
             for ns in (0, 5000, 145000, 1 << 40)]
    # ties: (4 w / p) an odd square, e.g. 195 K tiles over 56 tiles, between 7 and 8 pieces
    assert (195, 56, 512, 0) in cases and model(195, 56, 512, 0) == 8
    assert evaluate("split_pieces", cases, tmp_path) == [model(*c) for c in cases]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_fp32_pieces(tmp_path):
    """No more than 16 pieces, than stages of 32, than the workspace's bound; no rows, fewer rows than experts; and the
    count that was measured as the fastest."""
    cases = [(E, N, K, M) for E in (1, 3, 8, 64) for N in (0, 1, 2, 65, 130, 1000, 4096, 100000)
             for K in (8, 32, 40, 648, 4096, 28672) for M in (8, 136, 1024, 28672)]
    for (E, N, K, M), s in zip(cases, evaluate("gmm_f32_pieces", cases, tmp_path)):
        assert 1 <= s <= 16 and s <= (K + 31) // 32 and (s == 1 or (N > 0 and s * N * M <= 512 * 128 * 128)), (E, N, K, M, s)
    measured = [(8, 4096, 2048, 512), (8, 2000, 5632, 1024), (4, 130, 3584, 896), (8, 4096, 512, 2048)]
    assert evaluate("gmm_f32_pieces", measured, tmp_path) == [3, 3, 16, 1]
