"""fp32 grouped GEMMs on split operands: tile edges, remainders, empty experts, and operands with
infinities, NaN and values at the end of the range, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu

COUNTS = [0, 1, 63, 64, 65, 0, 127, 128, 129, 200, 7]
MODES = ["NN", "NT", "TN"]


def product(pkg, mode, a, b, off):
    return pkg.ops.gmm(a, b, off, trans_a=mode == "TN", trans_b=mode == "NT")


def operands(mode, N, K, M, E, dev, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(N, K, generator=g)
    b = torch.randn(*{"NN": (E, K, M), "NT": (E, M, K), "TN": (N, M)}[mode], generator=g)
    return a.to(dev), b.to(dev)


def reference(mode, a, b, counts, f=lambda t: t):
    """Per-expert float64 products of f(a) and f(b) on the CPU."""
    a, b, out, lo = f(a.double().cpu()), f(b.double().cpu()), [], 0
    for e, n in enumerate(counts):
        r = slice(lo, lo + n)
        lo += n
        out.append(a[r].T @ b[r] if mode == "TN" else a[r] @ (b[e] if mode == "NN" else b[e].T))
    return torch.stack(out) if mode == "TN" else torch.cat(out)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("K, M", [(8, 8), (40, 136), (520, 264), (136, 2048)])
def test_edges(pkg, dev, mode, K, M):
    E, N = len(COUNTS), sum(COUNTS)
    off = torch.tensor([0] + COUNTS, device=dev).cumsum(0)
    a, b = operands(mode, N, K, M, E, dev, K + M)
    got = product(pkg, mode, a, b, off).double().cpu()
    # the three dropped partial products are below 2^-24 of a product; a sum passes at most 12 accumulations
    # of 16 products in its block and one addition per block of 32, each within 2^-24 of the absolute sum
    red = max(COUNTS) if mode == "TN" else K
    bound = 2.0 ** -24 * (1 + 12 + (red + 31) // 32) * reference(mode, a, b, COUNTS, torch.abs)
    assert ((got - reference(mode, a, b, COUNTS)).abs() <= bound).all()


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("value, other", [(float("inf"), 1.0), (float("-inf"), 0.0), (float("nan"), 1.0),
                                          (torch.finfo(torch.float32).max, 2.0 ** -20)])
def test_non_finite_operands(pkg, dev, mode, value, other):
    """One extreme element in a, opposite an exactly representable one in b: infinities stay infinities."""
    counts, K, M = [70, 150], 72, 200
    off = torch.tensor([0] + counts, device=dev).cumsum(0)
    a, b = operands(mode, sum(counts), K, M, 2, dev, 11)
    a[100, 9] = value
    if mode == "TN":
        b[100] = other
    elif mode == "NN":
        b[1, 9] = other
    else:
        b[1, :, 9] = other
    got, ref = product(pkg, mode, a, b, off).double().cpu(), reference(mode, a, b, counts)
    assert torch.equal(got.isnan(), ref.isnan())
    assert torch.equal(got.isinf(), ref.isinf()) and torch.equal(got[got.isinf()], ref[ref.isinf()])
    finite = ref.isfinite()
    # 200 sequential additions at most (the fp32 MFMA's order), each within 2^-24 of the absolute sum
    mag = reference(mode, a, b, counts, torch.abs)
    assert ((got - ref).abs()[finite] <= 2.0 ** -24 * 200 * mag[finite]).all()
