"""The piece count of a split reduction (csrc/split_rule.h) against the same rule in whole numbers of Python: the
kernels of a split launch each come to it for themselves, so a tie may not hang on the rounding of a float."""
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
  long long es, k, t, slots, ns;
  while (std::scanf("%lld %lld %lld %lld %lld", &es, &k, &t, &slots, &ns) == 5)
    std::printf("%d\\n", gmoe::split_pieces(gmoe::split_ns_per_k_tile((int)es), k, t, slots, ns));
}
"""


def model(elem_bytes, k_tiles, tiles, slots, stream_ns):
    if tiles == 0:
        return 1
    most = min(slots // tiles, 8, k_tiles)
    if most < 2:
        return 1
    whole, per_piece = (420 if elem_bytes == 2 else 2100) * k_tiles, 26 * tiles
    s = max([2] + [n for n in range(2, most + 1) if (2 * n - 1) ** 2 * per_piece <= 4 * whole])
    return s if whole - max(whole // s, stream_ns) > 6000 + per_piece * s else 1


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_pieces(tmp_path):
    (tmp_path / "rule.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "rule")
    subprocess.check_call(["g++", "-O2", "-I" + CSRC, str(tmp_path / "rule.cpp"), "-o", exe])
    cases = [(es, k, t, slots, ns) for es in (2, 4) for k in (1, 2, 5, 15, 16, 39, 44, 64, 224, 896, 1 << 22)
             for t in (0, 1, 4, 31, 32, 56, 96, 128, 255, 256, 257, 100000) for slots in (2, 511, 512)
             for ns in (0, 5000, 145000, 1 << 40)]
    # ties: (4 w / p) an odd square, e.g. 39 K tiles in fp32 over 56 tiles, between 7 and 8 pieces
    assert (4, 39, 56, 512, 0) in cases and model(4, 39, 56, 512, 0) == 8
    out = subprocess.run([exe], input="\n".join("%d %d %d %d %d" % c for c in cases), text=True,
                         capture_output=True, check=True).stdout.split()
    assert [int(v) for v in out] == [model(*c) for c in cases]
