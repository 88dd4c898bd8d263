"""Capacity selection against a stable sort on the CPU, at the edges of its blocks of 1024 tokens and of
the 16384 tokens (kCapKeys * kCapThreads) whose keys stay in LDS.  Bit for bit: it moves values and computes none."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T, E", [(1, 3), (63, 5), (1024, 4), (1025, 7), (16384, 2), (16385, 3), (33000, 2)])
def test_edges(pkg, dev, dtype, T, E):
    gen = torch.Generator().manual_seed(T * 7 + E)
    probs = torch.rand(T, E, generator=gen) - 0.25
    probs[:, 1] = (probs[:, 1] * 8).round() / 8 + 0.0  # many equal keys; no negative zero
    probs[torch.rand(T, E, generator=gen) < 0.6] = 0.0
    probs[T // 2, E - 1] = float("inf")
    probs[T // 3, 0] = float("-inf")
    probs = probs.to(dtype)
    rmap = probs > 0
    for capacity in sorted({1, max(1, T // 5), max(1, T // 2), max(1, T - 1), T, T + 9}):
        for by_position in (False, True):
            keys = rmap.int() if by_position else probs.float()
            order = keys.sort(dim=0, descending=True, stable=True).indices[: min(capacity, T)]
            chosen = torch.zeros(T, E, dtype=torch.bool).scatter_(0, order, True)
            for pad in (False, True):
                keep = chosen if pad else chosen & rmap
                got_probs, got_map = pkg.ops.capacity_select(probs.to(dev), rmap.to(dev), capacity, by_position, pad)
                assert torch.equal(got_map.cpu(), keep)
                assert torch.equal(got_probs.cpu(), torch.where(keep, probs, torch.zeros((), dtype=dtype)))
