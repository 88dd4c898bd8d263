"""Weight gradients of narrow results, on each of the kernels that the estimate may choose for them; each launch is checked to
be the kernel meant."""
import pytest
import torch

from test_gmm_rows_gpu import on_kernel

pytestmark = pytest.mark.gpu

SMALL, LARGE, SHORT = "gmm_kernel", "gmm_dtl_kernel", "gmm_tn_kernel"  # 128x128, 256x256 and 128x256 tiles
CASES = [  # rows per expert, K, M, kernel
    ([2100] * 8, 256, 6144, LARGE),            # K under 512
    ([1000, 0, 1000, 1300, 900, 1100, 1000, 1000], 136, 4104, LARGE),  # ... ragged and under one tile, uneven, an empty expert
    ([2000, 0] * 6 + [700] * 12, 8712, 184, LARGE),  # M under 256, ragged, empty experts
    ([1561] * 24, 1544, 168, LARGE),
    ([160] * 6, 8192, 1016, LARGE),            # 132 tiles
    ([1700, 0, 900, 1500], 136, 4104, SHORT),  # 128x256 tiles, ragged, uneven, an empty expert
    ([900] * 24, 184, 872, SHORT),             # ... beyond 768 rows
    ([130] * 12, 2048, 136, SHORT),            # ... with few rows and one column tile, mostly padding
    ([100] * 4, 8200, 136, SHORT),
    ([31, 0, 1, 7], 136, 1000, SHORT),         # ... of a handful of rows
    ([1100] * 16, 616, 144, SMALL),            # M under 256
    ([1024, 1], 8200, 128, SMALL),             # ... the narrowest
    ([3000], 128, 136, SMALL),                 # a few tiles
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,K,M,kernel", CASES)
def test_weight_gradient_of_narrow_results(pkg, dev, counts, K, M, kernel, dtype):
    """Products of 16-bit operands are exact in fp32; n additions in fp32 in any order stay within n * 2^-24 of the
    sum of magnitudes (here of the order of sqrt(n) * 2^-24, bounded by 2^-14), the result's rounding within half a
    unit in the last place, which fp16 results below 2^-14 (products of a lone row) have at 2^-24."""
    g = torch.Generator().manual_seed(K + M)
    N, E = sum(counts), len(counts)
    a = torch.randn(N, K, generator=g).to(dtype)
    b = torch.randn(N, M, generator=g).to(dtype)
    print("case", counts[:2], E, K, M, dtype, flush=True)
    off = pkg.ops.expert_offsets_from_batch_sizes(torch.tensor(counts), dev)
    ad, bd = a.to(dev), b.to(dev)
    c = on_kernel(kernel, lambda: pkg.ops.gmm(ad, bd, off, trans_a=True))
    assert c.shape == (E, K, M) and c.dtype == dtype
    row = 0
    for e, n in enumerate(counts):
        x, y = a[row:row + n].float(), b[row:row + n].float()
        row += n
        want, terms = x.t() @ y, x.t().abs() @ y.abs()
        ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11  # half a unit of 8 or 11 bits
        bound = want.abs() * ulp + terms * 2.0 ** -14 + (2.0 ** -25 if dtype == torch.float16 else 0.0)
        err = (c[e].cpu().float() - want).abs()
        assert torch.all(err <= bound), (e, float((err - bound).max()))
