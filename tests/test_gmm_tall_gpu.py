"""The row-adaptive NN / NT tiles of up to 384 rows at their edges: experts of 0 and 1 rows, of one row more or less
than whole tiles of 320 and 384 rows and of several, reductions that end inside a round (64) and a stage (32) and are
shorter than the copies run ahead, columns that end inside a tile; plain, fp32 output, and with the activation and its
backward fused."""
import pytest
import torch

from test_gmm_rows_gpu import on_kernel

pytestmark = pytest.mark.gpu

# rows of the experts, K, F: F columns of d(act), 2 F of the forward
TALL = [
    ([0, 1, 319, 320, 321, 383, 384, 385, 0, 640, 767, 769, 1153, 1536, 700, 340], 1160, 904),
    ([384, 383, 0, 1152, 2305, 65, 1, 768, 769, 2000, 1100, 96, 700, 330, 384, 3000], 520, 520),
    ([1025, 1023, 1500, 0, 1, 2047, 960, 1024], 136, 1096),
    ([700, 0, 513, 640, 1, 1280, 961, 705], 2088, 2056),
]


@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,K,F", TALL)
def test_tall_edges(pkg, dev, dtype, rows, K, F, act):
    E, N, M = len(rows), sum(rows), 2 * F
    g = torch.Generator(device=dev).manual_seed(K + F)
    print("case", dtype, K, F, act, flush=True)
    off = torch.tensor([0] + rows, device=dev).cumsum(0)

    def rnd(*s, std=1.0):
        return torch.empty(*s, device=dev).normal_(0.0, std, generator=g).to(dtype)

    a, w1 = rnd(N, K), rnd(E, K, M, std=K ** -0.5)
    wt = rnd(E, F, K, std=K ** -0.5)

    def here(call):
        return on_kernel("gmm_rows_kernel", call)

    fc1, h = here(lambda: pkg.ops.gmm_glu(a, w1, off, act))
    plain = here(lambda: pkg.ops.gmm(a, w1, off))
    plain32 = here(lambda: pkg.ops.gmm(a, w1, off, out_dtype=torch.float32))
    dfc1 = here(lambda: pkg.ops.gmm_glu_bwd(a, wt, fc1, off, act))
    # plain NT of fewer than 768 rows per expert may go elsewhere; its sums have the same order there
    d = pkg.ops.gmm(a, wt, off, trans_b=True)
    d32 = pkg.ops.gmm(a, wt, off, trans_b=True, out_dtype=torch.float32)
    assert torch.equal(fc1, plain) and torch.equal(h, pkg.ops.glu_fwd(fc1, act))
    assert torch.equal(dfc1, pkg.ops.glu_bwd(d, fc1, act))
    assert torch.equal(plain, plain32.to(dtype)) and torch.equal(d, d32.to(dtype))
    # products of 16-bit values are exact in fp32; both sides round up to K additions of partial sums
    # of size about one (rows of a have norm sqrt(K), columns of w norm one): 2^-24 * sqrt(K) per
    # element typically, eight times that as the bound, and four times that for the tails of a normal sum
    tol = 8 * 2.0 ** -24 * K ** 0.5 * 4
    s = 0
    for e, n in enumerate(rows):
        x = a[s:s + n].double()
        for got, want in ((plain32, x @ w1[e].double()), (d32, x @ wt[e].double().t().contiguous())):
            err = (got[s:s + n].double() - want).abs().max().item() if n else 0.0
            assert err < tol, (e, n, err)
        s += n


# rows of the experts, K, F: averages of 4 to 90 rows, where a tile of each expert fills a round
FEW = [
    ([0, 1] * 15 + [0] * 30 + [95, 70, 60, 55], 264, 1024),  # most experts empty, some with one row
    ([4] * 64, 72, 512),
    ([63, 64, 65, 0, 127, 128, 129, 1] * 4, 1160, 1016),  # around one and two units (of 64 rows), ragged K and F
    ([95, 0, 200, 33, 7, 383, 1, 0], 520, 4088),
    ([17], 2056, 32760),
]


@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,K,F", FEW)
def test_few_rows_with_the_activation(pkg, dev, dtype, rows, K, F, act):
    """fc1 against float64, and the activation to the bits of its own kernel."""
    E, N = len(rows), sum(rows)
    assert N // E < 96
    g = torch.Generator(device=dev).manual_seed(K + F)
    print("case", dtype, K, F, act, flush=True)
    off = torch.tensor([0] + rows, device=dev).cumsum(0)
    a = torch.empty(N, K, device=dev).normal_(generator=g).to(dtype)
    w1 = torch.empty(E, K, 2 * F, device=dev).normal_(0.0, K ** -0.5, generator=g).to(dtype)
    fc1, h = on_kernel("gmm_rows_kernel", lambda: pkg.ops.gmm_glu(a, w1, off, act))
    assert torch.equal(h, pkg.ops.glu_fwd(fc1, act))
    # as above, and half a unit of 8 or 11 bits for the 16-bit result
    tol = 8 * 2.0 ** -24 * max(K, 64) ** 0.5 * 4
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    s = 0
    for e, n in enumerate(rows):
        if n:
            want = a[s:s + n].double() @ w1[e].double()
            assert ((fc1[s:s + n].double() - want).abs() - want.abs() * half).max().item() < tol + 2.0 ** -25, e
        s += n


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,K,F", [([32, 0, 95, 1], 128, 256), ([1], 136, 72), ([0, 0, 5, 0, 0, 0, 0, 0], 264, 520), ([70] * 8, 72, 136)])
def test_short_launches_with_the_activation(pkg, dev, dtype, rows, K, F):
    """One launch when they are called, two where a graph is captured: the same bits from both, in every replay."""
    g = torch.Generator(device=dev).manual_seed(K + F)
    off = torch.tensor([0] + rows, device=dev).cumsum(0)
    a = torch.empty(sum(rows), K, device=dev).normal_(generator=g).to(dtype)
    w1 = torch.empty(len(rows), K, 2 * F, device=dev).normal_(0.0, K ** -0.5, generator=g).to(dtype)
    print("case", dtype, rows, K, F, flush=True)
    fc1, h = on_kernel("gmm_rows_kernel", lambda: pkg.ops.gmm_glu(a, w1, off, "silu"))
    assert torch.equal(h, pkg.ops.glu_fwd(fc1, "silu"))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        pkg.ops.gmm(a, w1, off)
        pkg.ops.glu_fwd(fc1, "silu")
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fc1_graph, h_graph = pkg.ops.gmm_glu(a, w1, off, "silu")
    for _ in range(3):
        fc1_graph.zero_()
        h_graph.zero_()
        on_kernel("gmm_kernel", graph.replay)
        assert torch.equal(fc1_graph, fc1) and torch.equal(h_graph, h)
        assert torch.equal(pkg.ops.gmm_glu(a, w1, off, "silu")[1], h)


@pytest.mark.parametrize("K,M", [(8, 2056), (72, 2312), (4104, 2056), (1000, 2304)])
def test_tall_transposed(pkg, dev, K, M):
    """Plain NT of 768 rows per expert and more, with reductions of a few elements up to many rounds."""
    rows = [769, 1, 1537, 0, 2200, 384, 1151, 1300]
    g = torch.Generator(device=dev).manual_seed(K + M)
    off = torch.tensor([0] + rows, device=dev).cumsum(0)
    a = torch.empty(sum(rows), K, device=dev).normal_(generator=g).bfloat16()
    w = torch.empty(len(rows), M, K, device=dev).normal_(0.0, K ** -0.5, generator=g).bfloat16()
    got = on_kernel("gmm_rows_kernel", lambda: pkg.ops.gmm(a, w, off, trans_b=True, out_dtype=torch.float32))
    tol = 8 * 2.0 ** -24 * max(K, 64) ** 0.5 * 4  # as above
    s = 0
    for e, n in enumerate(rows):
        want = a[s:s + n].double() @ w[e].double().t().contiguous()
        assert n == 0 or (got[s:s + n].double() - want).abs().max().item() < tol, (e, n)
        s += n
