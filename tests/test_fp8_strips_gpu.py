"""The weight-streaming fp8 GEMM at the edges of its column strips (128 or 256 columns, by the number of items), of
its rounds over the compute units and of the row fragments that an item of the last round is cut into; each launch is
checked to have strips of the width meant."""
import pytest
import torch

from test_gmm_rows_gpu import on_kernel

pytestmark = pytest.mark.gpu

NARROW, WIDE = 1, 2  # column fragments of 32 per wavefront: strips of 128 and 256
CASES = {  # rows per expert, K, M, width
    "one stage, ragged columns, one expert of two chunks": ([1, 193], 64, 144, NARROW),
    "few items: their fragments shared out": ([0, 33, 192, 65, 300], 192, 400, NARROW),
    "one narrow strip": ([64], 128, 128, NARROW),
    "narrow strips, less than a round": ([32] * 20, 128, 1536, NARROW),
    "narrow strips, one expert's chunks beyond a round": ([20] * 15 + [400], 128, 2048, NARROW),
    "wide strips, less than a round": ([(37 * e) % 190 for e in range(24)], 192, 1424, WIDE),
    "wide strips, a round and a rest": ([(53 * e) % 201 for e in range(44)], 128, 1552, WIDE),
    "wide strips, three rounds, empty experts last": ([70] * 40 + [0, 0], 64, 4864, WIDE),
}


@pytest.mark.parametrize("fp8_rows", [False, True])
@pytest.mark.parametrize("name", CASES)
def test_fp8_strips_and_rounds(pkg, orc, dev, name, fp8_rows):
    """Products are exact; what remains is the result's bf16 rounding (2^-8 of it) and the order and precision of
    the sums, bounded by 2^-14 of the sum of the terms' magnitudes (the block-scaled MFMA's own precision)."""
    counts, K, M, width = CASES[name]
    bs = torch.tensor(counts, dtype=torch.int64)
    N, E = int(bs.sum()), len(counts)
    g = torch.Generator().manual_seed(N)
    a = torch.randn(N, K, generator=g).bfloat16()
    w = torch.randn(E, K, M, generator=g) / K ** 0.5
    print("case", name, fp8_rows, flush=True)
    off = pkg.ops.expert_offsets_from_batch_sizes(bs, dev)
    ad = a.float()
    if fp8_rows:
        aq, scales = pkg.ops.quantize_fp8_rows(a.to(dev))
        ad = orc.dequantize_fp8_rows(aq.cpu(), pkg.ops.row_scale_exponents(scales).cpu())
    for trans_b in (False, True):
        q, s = orc.quantize_fp8_block(w.transpose(1, 2).contiguous() if trans_b else w)
        wd = orc.dequantize_fp8_block(q, s)
        ac, qd, sd = a.to(dev), q.to(dev), s.to(dev)
        if fp8_rows:
            call = lambda: pkg.ops.gmm_fp8a(aq, scales, qd, sd, off, trans_b=trans_b)
        else:
            call = lambda: pkg.ops.gmm_fp8w(ac, qd, sd, off, trans_b=trans_b)
        c = on_kernel("gmm_fp8_skinny_kernel", call, ", %d" % width)
        ref = orc.gmm(ad, wd, bs, trans_b=trans_b)
        bound = ref.abs() * 2.0 ** -8 + orc.gmm(ad.abs(), wd.abs(), bs, trans_b=trans_b) * 2.0 ** -14
        err = (c.cpu().float() - ref).abs()
        assert torch.all(err <= bound), (trans_b, float((err - bound).max()))
