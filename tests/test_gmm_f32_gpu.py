"""fp32 grouped GEMMs on split operands: tile edges, remainders, empty experts, and operands with
infinities, NaN and values at either end of the range, against float64."""
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


@pytest.mark.parametrize("mode", ["NN", "NT"])
@pytest.mark.parametrize("counts, K, M", [([130], 3584, 128), ([0, 65, 0, 3], 1000, 136), ([520, 500, 490, 538], 2048, 512),
                                          ([1], 648, 8), ([37, 30, 41, 0], 1416, 2048)])
def test_pieces(pkg, dev, mode, counts, K, M):
    """Reductions cut into pieces, the last of them shorter, with a small element in the first piece and one in
    the last, in different rows; the same bits again."""
    E, N = len(counts), sum(counts)
    need = pkg._C.lib().gmoe_gmm_workspace_bytes(E, N, K, M, 0, mode == "NT", 0)
    assert need % (N * M * 4) == 0 and need >= 2 * N * M * 4
    off = torch.tensor([0] + counts, device=dev).cumsum(0)
    a, b = operands(mode, N, K, M, E, dev, K + M)
    a[0, 0] = a[N - 1, K - 1] = 2.0 ** -120
    got = product(pkg, mode, a, b, off)
    # as in test_edges, one more addition per piece; the pieces with a small element are products added one after
    # the other: 2^-24 of the absolute sum each
    pieces = need // (N * M * 4)
    bound = 2.0 ** -24 * (1 + 12 + (K + 31) // 32 + pieces + (K + pieces - 1) // pieces)
    ref, mag = reference(mode, a, b, counts), reference(mode, a, b, counts, torch.abs)
    assert ((got.double().cpu() - ref).abs() <= bound * mag).all()
    assert torch.equal(got, product(pkg, mode, a, b, off))


@pytest.mark.parametrize("mode", ["NN", "NT"])
def test_pieces_leave_rows_outside_the_groups(pkg, dev, mode):
    """An offset table over rows 40..170 of 300, as for some of the experts of a larger buffer: the other rows of
    the result stay as they were."""
    N, K, M, first, last = 300, 3584, 128, 40, 170
    L, nt = pkg._C.lib(), int(mode == "NT")
    a, b = operands(mode, N, K, M, 2, dev, 5)
    need = L.gmoe_gmm_workspace_bytes(2, N, K, M, 0, nt, 0)
    assert need >= 2 * N * M * 4
    off = torch.tensor([first, 100, last], device=dev)
    ws, c = torch.full((need // 4,), 1e30, device=dev), torch.full((N, M), 7.0, device=dev)
    assert L.gmoe_gmm(a.data_ptr(), b.data_ptr(), c.data_ptr(), off.data_ptr(), 2, N, K, M, 0, nt, 0, 0, ws.data_ptr(),
                      need, torch.cuda.current_stream().cuda_stream) == 0
    assert (c[:first] == 7.0).all() and (c[last:] == 7.0).all()
    want = pkg.ops.gmm(a[first:last].contiguous(), b, off - first, trans_b=bool(nt))
    # two orders of the same sums: 2^-24 of the absolute sum per addition, as in test_pieces, on either side
    mag = reference(mode, a[first:last], b, [60, 70], torch.abs)
    assert ((c[first:last] - want).double().cpu().abs() <= 2 * 2.0 ** -24 * (13 + 112 + 16) * mag).all()


@pytest.mark.parametrize("mode", ["NN", "NT"])
@pytest.mark.parametrize("room", [0, 0.5, 1, 2, 3.7, None])
def test_smaller_workspaces(pkg, dev, mode, room):
    """NULL, less than a piece, one, fewer pieces than wanted, all: as many as fit, and nothing is written behind."""
    counts, K, M = [37, 30, 41, 0], 1416, 2048
    E, N, L, nt = len(counts), sum(counts), pkg._C.lib(), int(mode == "NT")
    off = torch.tensor([0] + counts, device=dev).cumsum(0)
    a, b = operands(mode, N, K, M, E, dev, 3)
    piece, need = N * M * 4, L.gmoe_gmm_workspace_bytes(E, N, K, M, 0, nt, 0)
    assert need >= 4 * piece
    size = need if room is None else int(room * piece) // 4 * 4
    ws, c = torch.full((need // 4 + 1024,), 5.0, device=dev), torch.empty(N, M, device=dev)
    assert L.gmoe_gmm(a.data_ptr(), b.data_ptr(), c.data_ptr(), off.data_ptr(), E, N, K, M, 0, nt, 0, 0,
                      ws.data_ptr() if room != 0 else None, size, torch.cuda.current_stream().cuda_stream) == 0
    # what is used are whole pieces, two or more
    pieces = size // piece
    used = (ws != 5.0).nonzero()
    assert (len(used) == 0 and pieces < 2) or piece // 4 < int(used[-1]) + 1 <= pieces * piece // 4, (pieces, int(used[-1]))
    # as in test_pieces
    bound = 2.0 ** -24 * (1 + 12 + (K + 31) // 32 + 16)
    ref, mag = reference(mode, a, b, counts), reference(mode, a, b, counts, torch.abs)
    assert ((c.double().cpu() - ref).abs() <= bound * mag).all()


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


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("log2_a, log2_b", [(-103, 100), (-118, 100), (100, -118), (-124, 110), (110, -130),
                                            (-100, -20), (-20, -125), (-60, -80)])
def test_small_operands(pkg, dev, mode, log2_a, log2_b):
    """Magnitudes at which the planes of the split run out of exponent, opposite ordinary and large ones, and
    products that do: no less precise than fp32 products."""
    counts, K, M = [70, 150, 33], 72, 200
    off = torch.tensor([0] + counts, device=dev).cumsum(0)
    a, b = operands(mode, sum(counts), K, M, 3, "cpu", 12)
    a, b = (a * 2.0 ** log2_a).to(dev), (b * 2.0 ** log2_b).to(dev)
    a[90:120] = 0.0
    got, ref = product(pkg, mode, a, b, off).double().cpu(), reference(mode, a, b, counts)
    # one product after the other (the fp32 MFMA's order): the rounding of addition i has a variance of a third
    # of (2^-24)^2 times that of i products, together 2^-24 * sqrt(red / 6) of the result's norm; four times
    # that, and half the spacing of the subnormal numbers per addition
    red = max(counts) if mode == "TN" else K
    bound = 4 * 2.0 ** -24 * (red / 6) ** 0.5 * ref.norm() + red * 2.0 ** -150 * ref.numel() ** 0.5
    assert (got - ref).norm() <= bound, ((got - ref).norm() / bound).item()


@pytest.mark.parametrize("mode", MODES)
def test_one_small_element(pkg, dev, mode):
    """A single small element in a, the only one of its row (NN, NT) or column (TN) that is not zero."""
    counts, K, M = [70, 150], 72, 200
    off = torch.tensor([0] + counts, device=dev).cumsum(0)
    a, b = operands(mode, sum(counts), K, M, 2, dev, 13)
    if mode == "TN":
        a[:, 41] = 0.0
    else:
        a[170] = 0.0
    a[170, 41] = 1.2345678 * 2.0 ** -118
    got, ref = product(pkg, mode, a, b, off).double().cpu(), reference(mode, a, b, counts)
    got, ref = (got[1, 41], ref[1, 41]) if mode == "TN" else (got[170], ref[170])
    # one product, rounded once, and zeros
    assert ((got - ref).abs() <= 2.0 ** -24 * ref.abs() + 2.0 ** -149).all(), ((got - ref) / ref).abs().max().item()


@pytest.mark.parametrize("E, M", [(5, 264), (3, 40)])
def test_dw_beyond_2gib(pkg, dev, E, M):
    """dW of operands of 2 GiB and more on the fp32 MFMA kernels (256x256 and 128x128 tiles), one expert's rows
    longer than a buffer resource."""
    counts, K = [0, 135000, 1, 4000, 77][:E], 4096
    off = torch.tensor([0] + counts, device=dev).cumsum(0)
    g = torch.Generator(device=dev).manual_seed(M)
    a = torch.empty(sum(counts), K, device=dev).normal_(generator=g)
    b = torch.empty(sum(counts), M, device=dev).normal_(generator=g)
    assert a.numel() * 4 >= 1 << 31
    got, lo = product(pkg, "TN", a, b, off), 0
    for e, n in enumerate(counts):
        ref = a[lo:lo + n].double().t().contiguous() @ b[lo:lo + n].double()
        lo += n
        # as in test_small_operands
        assert (got[e].double() - ref).norm() <= 4 * 2.0 ** -24 * (n / 6 + 1) ** 0.5 * ref.norm()
