"""Argument forms of the native autograd nodes: what the tensor-level checks refuse, the slot of the loss
tracker that a layer index names, and writes in place on what a node returned."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture()
def routing_map(dev):
    return torch.tensor([[1, 0], [0, 1], [1, 0], [0, 1]], dtype=torch.bool, device=dev)


def test_rows_of_another_rank_are_refused(pkg, dev, routing_map):
    host = pkg._C.host()
    plan = pkg.ops.permute_plan(routing_map, 4, want_sorted=False)
    cube = torch.zeros(4, 8, 16, device=dev)
    scores = torch.rand(4, 2, 3, device=dev)
    calls = [
        lambda: host.permute_rows(cube, plan.dst_map, 4, False),
        lambda: pkg.unpermute(cube, plan.dst_map, (4, 8)),
        lambda: host.gate_fwd(cube, cube.view(8, 16, 4), torch.float32),
        lambda: host.seq_aux_loss(scores, scores > 0.5, 2, 2, 1, 0.01, "identity"),
        lambda: host.capacity_select(scores, scores > 0.5, 1, False, False),
    ]
    for call in calls:
        with pytest.raises((AssertionError, ValueError)):
            call()


@pytest.mark.parametrize("layer_idx, slot", [(None, None), (0, 2), (1, 0), (3, 2)])
def test_tracker_slot(pkg, dev, layer_idx, slot):
    """values[layer_idx - 1], counted from the end for layer 0; no entry without a layer index."""
    cfg = pkg.MoEConfig(hidden_size=64, num_moe_experts=4, moe_ffn_hidden_size=64, moe_router_topk=2,
                        moe_router_load_balancing_type="aux_loss", moe_aux_loss_coeff=0.01, num_layers=3,
                        params_dtype=torch.float32)
    router = pkg.GalvatronMoERouter(cfg, layer_idx=layer_idx, device=dev).train().router
    tracker = pkg.moe_utils.get_moe_layer_wise_logging_tracker()
    tracker.clear()
    router.routing(torch.randn(8, 1, 4, generator=torch.Generator().manual_seed(5)).to(dev).requires_grad_(True))
    values = tracker.pop("load_balancing_loss", {}).get("values")
    if slot is None:
        assert values is None
        return
    expected = torch.zeros(3)
    expected[slot] = router.last_aux_loss.item() / 0.01
    torch.testing.assert_close(values.cpu(), expected, rtol=1e-6, atol=0)


@pytest.mark.parametrize("transposed", [False, True])
def test_residual_is_not_written_in_place(pkg, dev, transposed):
    """The second output of PreRouterNorm is the input: writing it would change what the caller holds."""
    cfg = pkg.MoEConfig(hidden_size=64, num_moe_experts=4, moe_ffn_hidden_size=64, params_dtype=torch.float32)
    norm = pkg.PreRouterNorm(cfg, device=dev)
    x = torch.randn(4, 2, 64, generator=torch.Generator().manual_seed(1)).to(dev).requires_grad_(True)
    before = x.detach().clone()
    out, residual = norm(x.transpose(0, 1) if transposed else x)
    with pytest.raises(RuntimeError, match="modified inplace"):
        residual.add_(1.0)
    assert torch.equal(x.detach(), before)
    (out.sum() + (2 * residual).sum()).backward()
    assert x.grad is not None


@pytest.mark.parametrize("E", [16, 20, 24, 61])
def test_gate_records_one_node(pkg, dev, E):
    """Padding the router weight (20, 61 experts) is part of the launch: autograd records the projection and
    nothing else."""
    x = torch.randn(8, 64, device=dev, requires_grad=True)
    weight = torch.randn(E, 64, device=dev, requires_grad=True)
    before = (x * 1).grad_fn._sequence_nr()
    logits = pkg.router._GateProjection.apply(x, weight, torch.float32)
    after = (x * 1).grad_fn._sequence_nr()
    assert logits.grad_fn._sequence_nr() == before + 1 and after == before + 2
    (2 * logits).sum().backward()
    # sums of 8 and of at most 61 fp32 values of a few units, in another order
    torch.testing.assert_close(weight.grad, (2 * x.detach().sum(0)).expand(E, 64), rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(x.grad, (2 * weight.detach().sum(0)).expand(8, 64), rtol=1e-5, atol=1e-4)
