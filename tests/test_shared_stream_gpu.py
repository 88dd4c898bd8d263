"""The shared experts' stages on the side stream and on the current one, whichever the layer's size asks for: the bits
of the plain call in the output and in every gradient, also when the stages are called under another stream."""
import pytest
import torch

from test_shared_gpu import build

pytestmark = pytest.mark.gpu


def step(router, mlp, x, res, dy):
    xg = x.clone().requires_grad_(True)
    for p in list(router.parameters()) + list(mlp.parameters()):
        p.grad = None
    out = mlp(xg, res, *router(xg))
    out.backward(dy)
    return [out.detach(), xg.grad] + [p.grad for p in mlp.parameters()]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("min_us,side", [(0.0, True), (float("inf"), False), (None, False)])
def test_stage_streams_give_the_same_bits(pkg, dev, monkeypatch, dtype, min_us, side):
    _, router, mlp = build(pkg, dev, dtype, overlap=False)
    _, router2, mlp2 = build(pkg, dev, dtype, overlap=True)
    mlp2.load_state_dict(mlp.state_dict())
    router2.load_state_dict(router.state_dict())
    if min_us is not None:
        monkeypatch.setattr(pkg.SharedExpertMLP, "overlap_min_us", min_us)
    g = torch.Generator().manual_seed(7)
    x, res, dy = (torch.randn(96, 4, 256, generator=g).to(dtype).to(dev) for _ in range(3))
    shared = mlp2.shared_experts
    assert (shared._stage_stream(x) == pkg.SharedExpertMLP.stream) == side
    want = step(router, mlp, x, res, dy)
    for _ in range(3):
        got = step(router2, mlp2, x, res, dy)
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    # stages called under a stream that has not waited for the one they began on
    other = torch.cuda.Stream()
    with torch.no_grad():
        plain = shared(x)
        torch.cuda.synchronize()
        shared.pre_forward_comm(x * 1.0)
        with torch.cuda.stream(other):
            shared.linear_fc1_forward_and_act()
            shared.linear_fc2_forward()
            shared.post_forward_comm()
            late = shared.get_output()
            same = (late == plain).all()
    torch.cuda.synchronize()
    assert bool(same)


def test_line_between_the_streams(pkg, dev):
    """Few tokens of a small layer stay on the current stream; a layer whose weights or products take long does not."""
    _, _, small = build(pkg, dev, torch.bfloat16, overlap=True)
    _, _, large = build(pkg, dev, torch.bfloat16, overlap=True, E=32, H=1024, F=2048, Fs=2048, k=4)
    side = pkg.SharedExpertMLP.stream
    assert small.shared_experts._stage_stream(torch.empty(64, 1, 256, device=dev, dtype=torch.bfloat16)) != side
    few, many = (torch.empty(t, 1, 1024, device=dev, dtype=torch.bfloat16) for t in (1, 4096))
    assert large.shared_experts._stage_stream(few) != side and large.shared_experts._stage_stream(many) == side


def test_captured_side_stream_replays_the_eager_bits(pkg, dev, monkeypatch):
    monkeypatch.setattr(pkg.SharedExpertMLP, "overlap_min_us", 0.0)
    _, router, mlp = build(pkg, dev, torch.bfloat16, overlap=True)
    g = torch.Generator().manual_seed(8)
    x = torch.randn(64, 2, 256, generator=g).bfloat16().to(dev)
    with torch.no_grad():
        want = mlp(x, x, *router(x))
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                mlp(x, x, *router(x))
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = mlp(x, x, *router(x))
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
            torch.cuda.synchronize()


def test_small_layers_overlap_in_a_captured_graph(pkg, dev):
    """A layer that stays on the current stream when it is called takes the second one when it is captured, and replays the
    same bits; the smallest stay on one stream there too."""
    _, router, mlp = build(pkg, dev, torch.bfloat16, overlap=True, E=16, H=1024, F=512, Fs=1024, k=2)
    _, _, least = build(pkg, dev, torch.bfloat16, overlap=True)
    shared, side = mlp.shared_experts, pkg.SharedExpertMLP.stream
    g = torch.Generator().manual_seed(9)
    x = torch.randn(32, 2, 1024, generator=g).bfloat16().to(dev)
    little = torch.zeros(1, 1, 256, device=dev, dtype=torch.bfloat16)
    assert shared._stage_stream(x) != side
    with torch.no_grad():
        want = mlp(x, x, *router(x))
        warm = torch.cuda.Stream()
        warm.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(warm):
            for _ in range(2):
                mlp(x, x, *router(x))
        torch.cuda.current_stream().wait_stream(warm)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            chosen = shared._stage_stream(x), least.shared_experts._stage_stream(little)
            out = mlp(x, x, *router(x))
        assert chosen[0] == side and chosen[1] != side
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
            assert torch.equal(mlp(x, x, *router(x)), want)
