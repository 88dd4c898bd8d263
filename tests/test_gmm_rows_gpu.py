"""The row-adaptive NN / NT tiles and the TN tiles of short and long reductions at the edges of their chunks:
experts of 0 rows, of 1, of one row more or less than a unit (64), a tile (256) and two tiles, reductions that
end inside a stage, columns that end inside a tile; plain, fp32 output, and with the activation and its
backward fused.  Each launch is checked to be the kernel that the test is for."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [0, 1, 63, 64, 65, 127, 128, 129, 191, 193, 255, 256, 257, 320, 511, 513]
EDGES = [(1024, 1024, 4), (1160, 904, 4), (1544, 1096, 3), (520, 1024, 4)]  # K, F, times that ROWS are repeated


def on_kernel(kernel, call, form=""):
    """call(), with the only GEMM that it launches being `kernel`, its last template argument `form` (nothing is
    asked where the profiler sees no launch at all, as beside another profiler)."""
    from torch.profiler import ProfilerActivity, profile

    with profile(activities=[ProfilerActivity.CUDA]) as trace:
        out = call()
        torch.cuda.synchronize()
    names = [e.name for e in trace.events() if "gmoe::" in e.name and "gmm" in e.name]
    assert not names or (len(names) == 1 and "::%s<" % kernel in names[0] and form + ">(" in names[0]), names
    return out


@pytest.mark.parametrize("act", ["silu", "gelu"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K,F,times", EDGES)
def test_chunk_edges(pkg, dev, dtype, K, F, times, act):
    """Every size of expert `times` times: as often as it takes for F columns to be most of a round of tiles, short
    of which the launches go to smaller ones (48 experts, 1024 x 1024, us there and here: NT 41 / 44, backward 55 / 60)."""
    rows_of = ROWS * times
    E, N, M = len(rows_of), sum(rows_of), 2 * F
    g = torch.Generator(device=dev).manual_seed(K + F)
    print("case", dtype, K, F, act, flush=True)
    off = torch.tensor([0] + rows_of, device=dev).cumsum(0)

    def rnd(*s, std=1.0):
        return torch.empty(*s, device=dev).normal_(0.0, std, generator=g).to(dtype)

    a, w1 = rnd(N, K), rnd(E, K, M, std=K ** -0.5)
    wt = rnd(E, F, K, std=K ** -0.5)
    def rows(call):
        return on_kernel("gmm_rows_kernel", call)

    fc1, h = rows(lambda: pkg.ops.gmm_glu(a, w1, off, act))
    plain = rows(lambda: pkg.ops.gmm(a, w1, off))
    plain32 = rows(lambda: pkg.ops.gmm(a, w1, off, out_dtype=torch.float32))
    d = rows(lambda: pkg.ops.gmm(a, wt, off, trans_b=True))
    d32 = rows(lambda: pkg.ops.gmm(a, wt, off, trans_b=True, out_dtype=torch.float32))
    dfc1 = rows(lambda: pkg.ops.gmm_glu_bwd(a, wt, fc1, off, act))
    assert torch.equal(fc1, plain) and torch.equal(h, pkg.ops.glu_fwd(fc1, act))
    assert torch.equal(dfc1, pkg.ops.glu_bwd(d, fc1, act))
    assert torch.equal(plain, plain32.to(dtype)) and torch.equal(d, d32.to(dtype))
    # products of 16-bit values are exact in fp32; both sides round up to K additions of partial sums
    # of size about one (rows of a have norm sqrt(K), columns of w norm one): 2^-24 * sqrt(K) per
    # element typically, eight times that as the bound
    tol = 8 * 2.0 ** -24 * K ** 0.5 * 4
    s = 0
    for e, n in enumerate(rows_of):
        x = a[s:s + n].double()
        for got, want in ((plain32, x @ w1[e].double()), (d32, x @ wt[e].double().t().contiguous())):
            err = (got[s:s + n].double() - want).abs().max().item() if n else 0.0
            assert err < tol, (e, n, err)
        s += n


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K,M", [(1024, 512), (1160, 648), (136, 4104), (1160, 520)])
def test_short_reduction_edges(pkg, dev, dtype, K, M):
    """dW over 0, 1, a stage (32) more or less one, ... rows; output edges inside a tile."""
    rows = [0, 1, 31, 32, 33, 63, 64, 65, 95, 97, 128, 129, 7, 0, 300, 2]
    E, N = len(rows), sum(rows)
    g = torch.Generator(device=dev).manual_seed(K + M)
    print("case", dtype, K, M, flush=True)
    off = torch.tensor([0] + rows, device=dev).cumsum(0)
    a = torch.empty(N, K, device=dev).normal_(generator=g).to(dtype)
    b = torch.empty(N, M, device=dev).normal_(generator=g).to(dtype)
    got32 = on_kernel("gmm_tn_kernel", lambda: pkg.ops.gmm(a, b, off, trans_a=True, out_dtype=torch.float32))
    got = on_kernel("gmm_tn_kernel", lambda: pkg.ops.gmm(a, b, off, trans_a=True))
    assert torch.equal(got, got32.to(dtype))
    s = 0
    for e, n in enumerate(rows):
        want = a[s:s + n].double().t().contiguous() @ b[s:s + n].double()
        # exact products of values up to about 5 x 5, n fp32 additions: 2^-24 * 25 * n bounds each sum
        assert (got32[e].double() - want).abs().max().item() <= 2.0 ** -24 * 25 * n * 4
        s += n


STORE_NOW, STORE_NOW_STREAM, STORE_SPREAD = ", 0", ", 1", ", 2"  # how gmm_dtl_kernel stores a tile


def check_dw(pkg, dev, dtype, rows, K, M, form):
    E, N = len(rows), sum(rows)
    g = torch.Generator(device=dev).manual_seed(K + M)
    print("case", dtype, K, M, flush=True)
    off = torch.tensor([0] + rows, device=dev).cumsum(0)
    a = torch.empty(N, K, device=dev).normal_(generator=g).to(dtype)
    b = torch.empty(N, M, device=dev).normal_(generator=g).to(dtype)
    got32 = on_kernel("gmm_dtl_kernel", lambda: pkg.ops.gmm(a, b, off, trans_a=True, out_dtype=torch.float32), STORE_NOW)
    got = on_kernel("gmm_dtl_kernel", lambda: pkg.ops.gmm(a, b, off, trans_a=True), form)
    assert torch.equal(got, got32.to(dtype))
    s = 0
    for e, n in enumerate(rows):
        want = a[s:s + n].double().t().contiguous() @ b[s:s + n].double()
        # exact products of values up to about 5 x 5, n fp32 additions: 2^-24 * 25 * n bounds each sum; those of a
        # long reduction stay within a few sqrt(n)
        assert (got32[e].double() - want).abs().max().item() <= 2.0 ** -24 * 25 * min(n, 100 * n ** 0.5) * 4
        s += n


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K,M", [(1160, 904), (520, 4104)])
@pytest.mark.parametrize("rows", [[0, 1, 31, 3000, 32, 33, 95, 96, 97, 0, 0, 4097, 7, 2500, 65, 5000],
                                  [3000, 0, 287, 256, 288, 289, 257, 3500, 320, 384, 385, 0, 416, 417, 1, 5500]])
def test_long_reduction_edges(pkg, dev, dtype, rows, K, M):
    """dW on 256x256 tiles, whose copies run ahead into the next tile and whose results are stored under its MFMAs:
    experts with no rows, with less than the copies' three stages (96 rows), around the nine K tiles (of 32 rows)
    that the stores take and the fourths of the next tile that they are spread over, and with many, in turn;
    output edges inside a tile."""
    check_dw(pkg, dev, dtype, rows, K, M, STORE_SPREAD)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K,M", [(1160, 1096), (520, 4104)])
def test_medium_reduction_edges(pkg, dev, dtype, K, M):
    """dW on 256x256 tiles that are stored before the next one: around the copies' three stages (96 rows) and
    whole K tiles (32), empty experts in turn, and many rows; output edges inside a tile."""
    rows = [0, 1, 33, 159, 160, 161, 0, 191, 192, 193, 223, 225, 0, 900, 64, 700]
    check_dw(pkg, dev, dtype, rows, K, M, STORE_NOW)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_streamed_result_edges(pkg, dev, dtype):
    """dW on 256x256 tiles with a result of 290 MiB, stored past the caches, and operands of a twelfth of it, read
    beforehand: 85 rows per expert on average, empty experts in turn; output edges inside a tile."""
    rows = [0, 1, 33, 95, 96, 97, 0, 127, 160, 161, 64, 65, 0, 300, 31, 130]
    check_dw(pkg, dev, dtype, rows, 1160, 8200, STORE_NOW_STREAM)


@pytest.mark.parametrize("K,F", [(520, 4104), (896, 4096), (2056, 4104)])
def test_activation_backward_of_many_rows(pkg, dev, K, F):
    """512 rows per expert and more, where 256x256 tiles could be had: the fused backward is the backward of the
    separate product on those, to the bit."""
    counts = [513, 767, 1025, 640, 0, 1, 1300, 560]
    off = torch.tensor([0] + counts, device=dev).cumsum(0)
    g = torch.Generator(device=dev).manual_seed(K)

    def rnd(*s, std=1.0):
        return torch.empty(*s, device=dev).normal_(0.0, std, generator=g).bfloat16()

    a, wt, fc1 = rnd(sum(counts), K), rnd(len(counts), F, K, std=K ** -0.5), rnd(sum(counts), 2 * F)
    got = on_kernel("gmm_rows_kernel", lambda: pkg.ops.gmm_glu_bwd(a, wt, fc1, off, "silu"))
    d = on_kernel("gmm_kernel", lambda: pkg.ops.gmm(a, wt, off, trans_b=True))
    assert torch.equal(got, pkg.ops.glu_bwd(d, fc1, "silu"))
