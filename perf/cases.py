"""What this framework is timed on: the work its users have it do, through its public entry points.

Four kinds of work, told apart by a case's `kind`:

  step      one training step of an MoE layer: pre-router norm (optional), router, dispatch, experts,
            combine, residual, and the whole backward; gives the output, the gradients of the input
            and of every parameter, and the load-balancing loss
  forward   the same layer under no_grad: evaluation batches, prefill and decoding
  fp8       an expert shard on frozen block-scaled fp8 weights: the rows another rank sent, forward,
            with `grad` also the gradient of the rows
  move      `permute` / `unpermute` as free functions, with their backward

`listed()` spans the configurations in `configs.WORKLOADS` and what lies between and below them;
`draw()` draws from the same ranges.
"""
import importlib.util
import math
import os
import sys

import torch

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def package():
    """The framework (its folder has a hyphen, so it is loaded by path)."""
    name = "hetu_galvatron_amd"
    if name not in sys.modules:
        folder = os.path.join(os.getcwd(), "hetu-galvatron_amd")
        spec = importlib.util.spec_from_file_location(
            name, os.path.join(folder, "__init__.py"), submodule_search_locations=[folder])
        module = importlib.util.module_from_spec(spec)
        sys.modules[name] = module
        spec.loader.exec_module(module)
    return sys.modules[name]


# ---------------------------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------------------------

def layer(kind, tokens, hidden, ffn, experts, topk, dtype="bf16", batch=1, skew=0.0, norm=True, shared=0,
          dispatcher="allgather", balance="aux_loss", score="softmax", router_dtype="", z_loss=False,
          expert_bias=False, capacity=0.0, name=None):
    """One layer, tokens = sequence length * batch.  `skew`: spread of the experts' mean logits, in
    units of the logits' own spread; `shared`: width of the shared experts, which run on their own
    stream; `capacity`: capacity factor, the experts' blocks padded to it."""
    c = dict(kind=kind, tokens=tokens, hidden=hidden, ffn=ffn, experts=experts, topk=topk, dtype=dtype, batch=batch,
             skew=skew, norm=norm, shared=shared, dispatcher=dispatcher, balance=balance, score=score,
             router_dtype=router_dtype, z_loss=z_loss, expert_bias=expert_bias, capacity=capacity)
    return dict(c, name=name) if name else c


def shard(rows, hidden, ffn, experts, empty, fp8_rows, grad, name=None):
    c = dict(kind="fp8", rows=rows, hidden=hidden, ffn=ffn, experts=experts, empty=empty, fp8_rows=fp8_rows, grad=grad)
    return dict(c, name=name) if name else c


def move(tokens, hidden, experts, topk, dtype, name=None):
    c = dict(kind="move", tokens=tokens, hidden=hidden, experts=experts, topk=topk, dtype=dtype)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the test model: a debugging run or a unit test, all latency and launches
        layer("step", 64, 128, 256, 4, 2, batch=2, name="test_model_step"),
        # the small CPU-comparable configuration, trained in fp32
        layer("step", 2048, 512, 1024, 8, 2, dtype="fp32", batch=2, norm=False, name="tiny_step_fp32"),
        # pretraining of the Mixtral shape with four sequences per GPU: the headline configuration
        layer("step", 16384, 4096, 14336, 8, 2, batch=4, name="mixtral_step"),
        # fine-tuning of it on one packed batch of odd length, unevenly loaded experts, z-loss
        layer("step", 1531, 4096, 14336, 8, 2, skew=0.9, dispatcher="alltoall", z_loss=True,
              name="mixtral_finetune_step"),
        # pretraining of a fine-grained model: 64 small experts, top-8, shared experts beside them
        layer("step", 8192, 2048, 1408, 64, 8, shared=5632, name="finegrained_step"),
        # the DeepSeek-V3-shaped shard with bf16 weights: sigmoid gates, expert bias, fp32 router
        layer("step", 4096, 7168, 2048, 32, 8, balance="none", score="sigmoid", router_dtype="fp32", expert_bias=True,
              name="dsv3_shard_step"),
        # capacity factor with padded blocks, fp16, sequence-level loss
        layer("step", 2048, 1024, 2816, 16, 4, dtype="fp16", batch=4, skew=0.5, dispatcher="alltoall",
              balance="seq_aux_loss", capacity=1.25, name="capacity_step_fp16"),
        # decoding with the Mixtral shape: a few tokens, every expert's weights
        layer("forward", 13, 4096, 14336, 8, 2, name="mixtral_decode"),
        # prefill / evaluation of one prompt on the fine-grained model
        layer("forward", 1111, 2048, 1408, 64, 8, skew=0.3, shared=5632, name="finegrained_prefill"),
        # the fp8 shard as configured: frozen fp8 weights under a trained trunk, bf16 rows
        shard(4096, 7168, 2048, 32, 2, False, True, name="fp8_shard_step"),
        # serving on it: one decoding batch's rows, quantised as well
        shard(414, 7168, 2048, 32, 2, True, False, name="fp8_shard_decode"),
        # dispatch and combine alone, for a caller with experts of its own
        move(8192, 2048, 64, 8, "bf16", name="dispatch_combine"),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _width(rng, low, high):
    """A model width: mostly a multiple of 128, sometimes only of 32 or 16."""
    step = rng.choice((128, 128, 128, 128, 32, 16))
    return max(step, int(round(_log(rng, low, high) / step)) * step)


def _cost(c):
    """Comparable cost: time at the rates of the matrix cores and of the memory."""
    w = work(c)
    return w["flops"] * (16 if c.get("dtype") == "fp32" else 1) / 1.2e15 + w["bytes"] / 4e12


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(("step", "step", "step", "step", "forward", "forward", "fp8", "fp8", "move"))
        experts = rng.choice((4, 6, 8, 8, 16, 24, 32, 60, 64, 64))
        topk = min(rng.choice((1, 2, 2, 4, 6, 8, 8)), experts // 2)
        if kind == "fp8":
            c = shard(_log(rng, 32, 8192), 128 * _log(rng, 8, 56), 128 * _log(rng, 4, 24), rng.choice((8, 16, 32)),
                      rng.choice((0, 1, 2)), rng.random() < 0.5, rng.random() < 0.6)
        elif kind == "move":
            c = move(_log(rng, 16, 16384), _width(rng, 128, 7168), experts, topk, rng.choice(("bf16", "bf16", "fp16", "fp32")))
        else:
            batch = rng.choice((1, 1, 1, 2, 4))
            tokens = _log(rng, 16, 16384) if kind == "step" else _log(rng, 1, 4096)
            tokens = max(1, tokens // batch) * batch
            hidden, ffn = _width(rng, 128, 7168), _width(rng, 128, 14336)
            balance = rng.choice(("aux_loss", "aux_loss", "none", "seq_aux_loss"))
            sigmoid = rng.random() < 0.25
            c = layer(kind, tokens, hidden, ffn, experts, topk,
                      dtype=rng.choice(("bf16", "bf16", "bf16", "bf16", "bf16", "fp16", "fp32")), batch=batch,
                      skew=rng.choice((0.0, 0.0, 0.3, 0.9)), norm=rng.random() < 0.75,
                      shared=_width(rng, 256, 8192) if rng.random() < 0.25 else 0,
                      dispatcher=rng.choice(("allgather", "alltoall")), balance=balance,
                      score="sigmoid" if sigmoid else "softmax", router_dtype=rng.choice(("", "", "fp32")),
                      z_loss=rng.random() < 0.25, expert_bias=sigmoid and rng.random() < 0.5)
            if rng.random() < 0.12 and tokens * topk >= 2 * experts:
                c.update(dispatcher="alltoall", capacity=rng.choice((1.0, 1.25, 2.0)), shared=0)
        weights = 3.0 * c["experts"] * c["hidden"] * c.get("ffn", 0)
        if weights < 1.45e9 and _cost(c) <= most:
            return c


# ---------------------------------------------------------------------------------------------
# One case on the GPU
# ---------------------------------------------------------------------------------------------

def _normal(shape, std, dtype, gen):
    t = torch.empty(shape, device="cuda", dtype=dtype)
    return t.normal_(0.0, std, generator=gen)


def prepare(case, seed):
    pkg = package()
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return {"step": _prepare_layer, "forward": _prepare_layer, "fp8": _prepare_shard, "move": _prepare_move}[
        case["kind"]](pkg, case, seed, gen)


def _prepare_layer(pkg, c, seed, gen):
    dtype, H = DTYPES[c["dtype"]], c["hidden"]
    cfg = pkg.MoEConfig(
        hidden_size=H, num_moe_experts=c["experts"], moe_ffn_hidden_size=c["ffn"], moe_router_topk=c["topk"],
        moe_router_load_balancing_type=c["balance"], moe_router_score_function=c["score"],
        moe_router_dtype=c["router_dtype"] or None, moe_aux_loss_coeff=0.0 if c["balance"] == "none" else 0.01,
        moe_z_loss_coeff=1e-3 if c["z_loss"] else None, moe_router_enable_expert_bias=c["expert_bias"],
        moe_token_dispatcher_type=c["dispatcher"], moe_expert_capacity_factor=c["capacity"] or None,
        moe_pad_expert_input_to_capacity=bool(c["capacity"]),
        moe_shared_expert_intermediate_size=c["shared"] or None, moe_shared_expert_overlap=bool(c["shared"]),
        params_dtype=dtype)
    train = c["kind"] == "step"
    router = pkg.GalvatronMoERouter(cfg, device="cuda").train(train)
    mlp = pkg.GalvatronMoEMLP(cfg, device="cuda").train(train)
    norm = pkg.PreRouterNorm(cfg, device="cuda").train(train) if c["norm"] else None
    x = _normal((c["tokens"] // c["batch"], c["batch"], H), 1.0, dtype, gen)
    with torch.no_grad():
        for p in list(router.parameters()) + list(mlp.parameters()):
            p.normal_(0.0, cfg.init_method_std, generator=gen)
        if c["skew"]:
            # hidden states share a component, and the experts' router rows lean on it by different
            # amounts: uneven loads without any token being special
            lean = torch.empty(c["experts"], device="cuda").normal_(0.0, 1.0, generator=gen)
            common = torch.empty(H, device="cuda").normal_(0.0, 1.0, generator=gen)
            x += (0.5 * common).to(dtype)
            reach = c["skew"] * cfg.init_method_std * math.sqrt(H) / (0.5 * float(H))
            router.router.weight += (reach * lean[:, None] * common[None, :]).to(dtype)
        if c["expert_bias"]:
            router.router.expert_bias.normal_(0.0, 0.02, generator=gen)
    state = dict(case=c, router=router, mlp=mlp, norm=norm, x=x)
    if train:
        x.requires_grad_(True)
        state["dy"] = _normal(x.shape, 1.0, dtype, gen)
        state["params"] = [p for m in (norm, router, mlp) if m is not None for p in m.parameters()]
    return state


def _prepare_shard(pkg, c, seed, gen):
    E, H, F = c["experts"], c["hidden"], c["ffn"]
    cfg = pkg.MoEConfig(hidden_size=H, num_moe_experts=E, moe_ffn_hidden_size=F)
    mlp = pkg.GroupedMLP(E, cfg, device="cuda")
    with torch.no_grad():
        mlp.weight1.normal_(0.0, cfg.init_method_std, generator=gen)
        mlp.weight2.normal_(0.0, cfg.init_method_std, generator=gen)
    fp8 = pkg.Fp8GroupedMLP(mlp, fp8_activations=c["fp8_rows"])
    del mlp
    x = _normal((c["rows"], H), 1.0, torch.bfloat16, gen)
    counts = pkg.configs.multinomial_counts(c["rows"], E, seed=seed, empty=c["empty"]).cuda()
    state = dict(case=c, fp8=fp8, x=x, counts=counts)
    if c["grad"]:
        x.requires_grad_(True)
        state["dy"] = _normal((c["rows"], H), 1.0, torch.bfloat16, gen)
    return state


def _prepare_move(pkg, c, seed, gen):
    T, H, E, k, dtype = c["tokens"], c["hidden"], c["experts"], c["topk"], DTYPES[c["dtype"]]
    x = _normal((T, H), 1.0, dtype, gen).requires_grad_(True)
    scores, chosen = _normal((T, E), 1.0, torch.float32, gen).topk(k, dim=1)
    gates = torch.zeros((T, E), device="cuda", dtype=dtype).scatter_(1, chosen, scores.softmax(1).to(dtype))
    routing_map = torch.zeros((T, E), device="cuda", dtype=torch.bool).scatter_(1, chosen, True)
    return dict(case=c, permute=pkg.permute, unpermute=pkg.unpermute, x=x, gates=gates.requires_grad_(True),
                routing_map=routing_map, dy=_normal((T, H), 1.0, dtype, gen))


def _layer_forward(s, x):
    hidden, residual = s["norm"](x) if s["norm"] is not None else (x, None)
    probs, routing_map = s["router"](hidden)
    return s["mlp"](hidden, residual, probs, routing_map), probs


def run(s):
    c, x = s["case"], s["x"]
    if c["kind"] == "step":
        x.grad = None
        for p in s["params"]:
            p.grad = None
        out, _ = _layer_forward(s, x)
        out.backward(s["dy"])
        aux = s["router"].router.last_aux_loss
        return [out.detach(), x.grad] + [p.grad for p in s["params"]] + ([] if aux is None else [aux])
    if c["kind"] == "forward":
        with torch.no_grad():
            return list(_layer_forward(s, x))
    if c["kind"] == "fp8":
        if not c["grad"]:
            with torch.no_grad():
                return s["fp8"](x, s["counts"])[0]
        x.grad = None
        out, _ = s["fp8"](x, s["counts"])
        out.backward(s["dy"])
        return [out.detach(), x.grad]
    x.grad = s["gates"].grad = None
    permuted, mapping = s["permute"](x, s["routing_map"], num_out_tokens=c["tokens"] * c["topk"])
    out = s["unpermute"](permuted, mapping, x.shape, probs=s["gates"], routing_map=s["routing_map"])
    out.backward(s["dy"])
    return [permuted.detach(), mapping, out.detach(), x.grad, s["gates"].grad]


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without, and how far another correct implementation may lie
# ---------------------------------------------------------------------------------------------

def work(c):
    E, H = c["experts"], c["hidden"]
    if c["kind"] == "fp8":
        N, F = c["rows"], c["ffn"]
        busy = (E - c["empty"]) * (1.0 - (1.0 - 1.0 / (E - c["empty"])) ** N)
        flops, nbytes = 6.0 * N * H * F, 3.0 * busy * H * F + 4.0 * N * H
        if c["grad"]:
            flops, nbytes = 2 * flops, nbytes + 4.0 * N * H
        return {"bytes": nbytes, "flops": flops}
    size = 4 if c["dtype"] == "fp32" else 2
    T, k = c["tokens"], c["topk"]
    if c["kind"] == "move":
        # forward: x, the permuted rows, the output; backward: dy, dx; the gates, their gradient, the map
        return {"bytes": size * (4.0 * T * H + T * k * H) + T * E * (2 * size + 1) + 8.0 * T * k,
                "flops": 5.0 * T * k * H}
    N, F = T * k, c["ffn"]
    busy = E * (1.0 - (1.0 - k / E) ** T)
    flops = 6.0 * N * H * F + 6.0 * T * H * c["shared"] + 2.0 * T * H * E
    weights = size * (3.0 * busy * H * F + 3.0 * H * c["shared"] + E * H)
    nbytes = weights + size * 2.0 * T * H
    if c["kind"] == "step":
        all_weights = size * (3.0 * E * H * F + 3.0 * H * c["shared"] + E * H)
        flops, nbytes = 3 * flops, nbytes + all_weights + size * 2.0 * T * H
    return {"bytes": nbytes, "flops": flops}


def tolerance(c):
    """About four times what the path shows against itself with wider types (the same layer in fp32 on
    the same values, fp32 against fp64): bf16 steps 2e-3 (outputs) to 5e-3 (gate gradient), fp16 steps
    2e-4 to 7e-4, fp32 steps 8e-7 and more with longer sums, the fp8 shard 3.5e-3.  A quantised row
    moves by an fp8 step when its bf16 value moves by one place, hence the wider bound there."""
    if c["kind"] == "move":
        return {"rel": {"bf16": 4e-3, "fp16": 5e-4, "fp32": 1e-6}[c["dtype"]]}
    if c["kind"] == "fp8":
        return {"rel": 2e-2 if c["fp8_rows"] else 1.4e-2}
    return {"rel": {"bf16": 2e-2, "fp16": 3e-3, "fp32": 1e-5}[c["dtype"]]}
