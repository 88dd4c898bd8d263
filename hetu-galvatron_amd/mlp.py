"""Expert MLPs with the reference's interface (galvatron/core/runtime/moe/mlp.py).

`GroupedMLP` (mlp.py:26-126): weight1 [H, E*2F] viewed [E,H,2F] (gate half first), weight2 [E*F, H]
viewed [E,F,H]; forward(permuted [N,H], tokens_per_expert [E]) -> (out [N,H], None) computed as
grouped GEMM -> gated activation -> grouped GEMM on the HIP kernels.
`SharedExpertMLP` (mlp.py:215-400): a dense gated MLP over all tokens with the reference's
parameters (`linear_fc1.weight [2Fs,H]`, `linear_fc2.weight [H,Fs]`, optional `gate_weight [1,H]`),
run as one group on the grouped kernels, optionally on its own stream beside the routed experts.
"""
from __future__ import annotations

import contextlib

import torch
import torch.nn.functional as F
from torch.nn.parameter import Parameter

from . import _C, ops
from .config import MoEConfig
from .grouped_gemm import ops as gg_ops


def glu(y: torch.Tensor, act: str = "silu", fp8_input_store: bool = False) -> torch.Tensor:
    """act(y[:, :F]) * y[:, F:]  (mlp.py:52-57; backward transformer/fused_kernels.py:157-162).
    `fp8_input_store`: the input is kept as float8_e4m3fn for the backward (SwiGLUFunction with
    fp8_input_store, transformer/fused_kernels.py:190-204): a quarter (fp32) or half (16-bit) of the saved
    bytes, the gradient computed on the rounded input."""
    shape = y.shape
    out = _C.host().glu(y.reshape(-1, shape[-1]).contiguous(), act, fp8_input_store)
    return out.view(*shape[:-1], shape[-1] // 2)


def swiglu(y: torch.Tensor) -> torch.Tensor:
    """transformer/fused_kernels.py:142-145."""
    return glu(y, "silu")


class _BiasRows(torch.autograd.Function):
    """x [N,M] + bias [M] row by row (x None: the bias alone as `num_rows` rows); the bias gradient
    is the column sum of the incoming gradient."""

    @staticmethod
    def forward(ctx, x, bias, num_rows):
        ctx.has_x = x is not None
        ctx.bias_shape = bias.shape
        return ops.bias_rows(None if x is None else x.contiguous(), bias.contiguous(), num_rows)

    @staticmethod
    def backward(ctx, grad):
        grad = grad.contiguous()
        grad_bias = ops.bias_rows_bwd(grad).view(ctx.bias_shape) if ctx.needs_input_grad[1] else None
        return (grad if ctx.has_x else None), grad_bias, None


def add_bias(x: torch.Tensor, bias: torch.Tensor) -> torch.Tensor:
    """`intermediate_parallel + bias_parallel` (transformer/mlp.py:132-133) on rows [..., M]."""
    shape = x.shape
    return _BiasRows.apply(x.reshape(-1, shape[-1]), bias, None).view(shape)


def expand_bias(bias: torch.Tensor, num_rows: int) -> torch.Tensor:
    """`output_bias.expand_as(output)` (moe/mlp.py:203) as rows of their own, [num_rows, M]."""
    return _BiasRows.apply(None, bias, num_rows)


def bias_swiglu_impl(input, bias, fp8_input_store=False):
    """transformer/fused_kernels.py:207-216: swiglu(input + bias), the sum rounded to the input's
    dtype as the reference's `y + bias` is."""
    if bias is not None:
        input = add_bias(input, bias)
    return glu(input, "silu", fp8_input_store)


class _FusedGatedExperts:
    """out = gmm(act(gmm(x, w1)[:, :F]) * gmm(x, w1)[:, F:], w2) with the activation fused into the
    first GEMM's epilogue and its backward into the epilogue of the d(act) GEMM
    (same math, op by op, as moe/mlp.py:106-112 and its autograd)."""

    # The fused d(act) GEMM + activation backward gives the same bits as the two launches.  Its
    # epilogue reads fc1 and writes d(fc1) (4 bytes of HBM traffic per accumulator) while the matrix
    # cores of that workgroup's CU idle, which the separate activation-backward kernel at HBM speed
    # does not make up for (us fused / apart: 8 experts of 4096 rows, 4096 x 14336 3202 / 3642, of 383 369 / 385; 64 of
    # 1024, 2048 x 1408 421 / 508; 32 of 1024, 7168 x 2048 776 / 846), and it never materialises d(act) (0.94 GB at the
    # first of these).
    fuse_backward = True

    @staticmethod
    def apply(x, w1, w2, batch_sizes, act):
        offsets = ops.expert_offsets_from_batch_sizes(batch_sizes, x.device)
        return _C.host().gated_experts(x, w1, w2, offsets, act, _FusedGatedExperts.fuse_backward)


def fused_gated_experts(x, w1, w2, batch_sizes, act: str = "silu"):
    """x [N,H], w1 [E,H,2F], w2 [E,F,H], batch_sizes [E] -> [N,H]."""
    return _FusedGatedExperts.apply(x, w1, w2, batch_sizes, act)


def fp8_gated_experts(x, w1_q, w1_scale, w2_q, w2_scale, batch_sizes, act: str = "silu",
                      fp8_activations: bool = False):
    """x [N,H] bf16; (w1_q [E,H,2F], w1_scale) and (w2_q [E,F,H], w2_scale) from
    ops.quantize_fp8_block; batch_sizes [E] -> [N,H] bf16.  `fp8_activations`: the rows entering each
    of the four products are quantised to fp8 as well (ops.quantize_fp8_rows) and the products run on
    the fp8 MFMA; off by default, where the bf16 rows are multiplied with the exactly widened weights.
    The weights are frozen: the gradient is that of x only, its products read the same fp8 tensors with the
    transposed-operand flag."""
    offsets = ops.expert_offsets_from_batch_sizes(batch_sizes, x.device)
    return _C.host().fp8_gated_experts(x, w1_q, w1_scale, w2_q, w2_scale, offsets, act, fp8_activations)


def _act_name(config: MoEConfig) -> str:
    if config.activation_func in (F.silu, "silu", "swiglu"):
        return "silu"
    if config.activation_func in (F.gelu, "gelu", "geglu"):
        return "gelu"
    raise ValueError("Activation function must be silu or gelu when using GroupedMLP.")


class GroupedMLP(torch.nn.Module):
    """All local experts in two grouped GEMMs."""

    def __init__(self, num_local_experts: int, config: MoEConfig, tp_of_ep_group=None,
                 layer_idx: int = None, device=None):
        super().__init__()
        self.config = config
        self.num_local_experts = num_local_experts
        assert config.add_bias_linear is False, \
            "bias not supported in Grouped GEMM yet, please set '--disable-bias-linear' instead."
        assert tp_of_ep_group is None, "expert tensor parallelism needs collectives (single GPU build)"
        assert config.gated_linear_unit, "GroupedMLP here implements the gated (SwiGLU / GeGLU) MLP"
        self.act = _act_name(config)
        device = torch.cuda.current_device() if device is None else device
        fc1_out = config.moe_ffn_hidden_size * num_local_experts * 2
        fc2_in = config.moe_ffn_hidden_size * num_local_experts
        self.weight1 = Parameter(torch.empty(config.hidden_size, fc1_out, device=device,
                                             dtype=config.params_dtype))
        self.weight2 = Parameter(torch.empty(fc2_in, config.hidden_size, device=device,
                                             dtype=config.params_dtype))
        self.layer_idx = layer_idx
        # True: activation fused into the GEMM epilogues; False: the reference's three-op sequence
        self.fuse_activation = True
        self.reset_parameters()

    def reset_parameters(self):
        std = self.config.init_method_std
        torch.nn.init.normal_(self.weight1, mean=0.0, std=std)
        torch.nn.init.normal_(self.weight2, mean=0.0, std=std)

    def forward(self, permuted_local_hidden_states: torch.Tensor, tokens_per_expert: torch.Tensor):
        E, H = self.num_local_experts, self.config.hidden_size
        w1 = self.weight1.view(E, H, -1)
        w2 = self.weight2.view(E, -1, H)
        if permuted_local_hidden_states.nelement() != 0 and self.fuse_activation:
            fc2_output = fused_gated_experts(permuted_local_hidden_states, w1, w2, tokens_per_expert,
                                             self.act)
        elif permuted_local_hidden_states.nelement() != 0:
            fc1_output = gg_ops.gmm(permuted_local_hidden_states, w1, tokens_per_expert, trans_b=False)
            intermediate = glu(fc1_output, self.act)
            fc2_output = gg_ops.gmm(intermediate, w2, tokens_per_expert, trans_b=False)
        else:
            # no token for the local experts: keep the parameters in the graph (mlp.py:113-124)
            h = torch.matmul(permuted_local_hidden_states, self.weight1.view(H, -1))
            half = h.shape[-1] // 2
            h = F.silu(h[:, :half]) * h[:, half:]
            fc2_output = torch.matmul(h, self.weight2.view(-1, H))
        return fc2_output, None


class Fp8GroupedMLP(torch.nn.Module):
    """GroupedMLP with frozen, block-scaled fp8 (e4m3) expert weights: same forward signature,
    gradients flow to the input only.  The reference has the fp8 expert path commented out
    (mlp.py:164-184); the weight format is the one of ops.quantize_fp8_block."""

    def __init__(self, mlp: GroupedMLP, fp8_activations: bool = False):
        super().__init__()
        self.config = mlp.config
        self.num_local_experts = mlp.num_local_experts
        self.act = mlp.act
        # also quantise the rows entering each product and run them on the fp8 MFMA (see ops.gmm_fp8a)
        self.fp8_activations = fp8_activations
        E, H = mlp.num_local_experts, mlp.config.hidden_size
        with torch.no_grad():
            w1_q, w1_s = ops.quantize_fp8_block(mlp.weight1.detach().view(E, H, -1))
            w2_q, w2_s = ops.quantize_fp8_block(mlp.weight2.detach().view(E, -1, H))
        for name, t in (("weight1_q", w1_q), ("weight1_scale", w1_s), ("weight2_q", w2_q),
                        ("weight2_scale", w2_s)):
            self.register_buffer(name, t)

    def forward(self, permuted_local_hidden_states: torch.Tensor, tokens_per_expert: torch.Tensor):
        if permuted_local_hidden_states.nelement() == 0:
            return permuted_local_hidden_states.new_zeros(permuted_local_hidden_states.shape), None
        out = fp8_gated_experts(permuted_local_hidden_states, self.weight1_q, self.weight1_scale,
                                self.weight2_q, self.weight2_scale, tokens_per_expert, self.act,
                                self.fp8_activations)
        return out, None


class _Linear(torch.nn.Module):
    """`weight [out, in]`, y = x @ weight^T, the layout of the reference's expert
    Column/RowParallelLinear (tensor_parallel/layers.py:547-988) at tensor-parallel size 1.  With
    `config.add_bias_linear` it carries `bias [out]` (zero-initialised, as there) and, like those
    layers under `skip_bias_add=True` (transformer/mlp.py:71, 87), does not add it: the caller does."""

    def __init__(self, in_features: int, out_features: int, config: MoEConfig, device):
        super().__init__()
        self.weight = Parameter(torch.empty(out_features, in_features, device=device,
                                            dtype=config.params_dtype))
        torch.nn.init.normal_(self.weight, mean=0.0, std=config.init_method_std)
        if config.add_bias_linear:
            self.bias = Parameter(torch.zeros(out_features, device=device, dtype=config.params_dtype))
        else:
            self.register_parameter("bias", None)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        # one group holding every row: the grouped GEMM with the transposed-operand flag; the
        # one-entry offset table lives on the device and is built once per row count
        return gg_ops.gmm(x, self.weight.unsqueeze(0), ops.one_group(x.shape[0], x.device), trans_b=True)


class ExpertMLP(torch.nn.Module):
    """One expert of SequentialMLP: linear_fc1 [2F, H] (gate rows first, then up rows), gated
    activation, linear_fc2 [H, F]  (transformer/mlp.py:23-134 with is_expert=True)."""

    def __init__(self, config: MoEConfig, device=None):
        super().__init__()
        assert config.gated_linear_unit
        self.act = _act_name(config)
        H, Fe = config.hidden_size, config.moe_ffn_hidden_size
        self.linear_fc1 = _Linear(H, 2 * Fe, config, device)
        self.linear_fc2 = _Linear(Fe, H, config, device)

    def forward(self, hidden_states: torch.Tensor):
        """Returns (output, output_bias): with `add_bias_linear` the fc1 bias is added in front of the
        activation and the fc2 bias is handed back un-added, [H] (transformer/mlp.py:104-138)."""
        fc2_bias = self.linear_fc2.bias
        if hidden_states.shape[0] == 0:
            keep = self.linear_fc1.weight.sum() + self.linear_fc2.weight.sum()
            if self.linear_fc1.bias is not None:
                keep = keep + self.linear_fc1.bias.sum()
            return hidden_states.new_zeros(hidden_states.shape) + 0.0 * keep, fc2_bias
        fc1 = self.linear_fc1(hidden_states)
        if self.linear_fc1.bias is not None:
            fc1 = add_bias(fc1, self.linear_fc1.bias)
        return self.linear_fc2(glu(fc1, self.act)), fc2_bias


class SequentialMLP(torch.nn.Module):
    """The experts one after the other, each on its slice of the permuted rows (mlp.py:128-211):
    `local_experts[i].linear_fc1.weight [2F,H]`, `.linear_fc2.weight [H,F]`."""

    def __init__(self, num_local_experts: int, config: MoEConfig, tp_of_ep_group=None,
                 tp_and_ep_group=None, layer_idx: int = None, device=None):
        super().__init__()
        assert tp_of_ep_group is None and tp_and_ep_group is None, \
            "expert tensor parallelism needs collectives (single GPU build)"
        self.config = config
        self.add_bias = config.add_bias_linear
        self.num_local_experts = num_local_experts
        device = torch.cuda.current_device() if device is None else device
        self.local_experts = torch.nn.ModuleList(
            [ExpertMLP(config, device=device) for _ in range(num_local_experts)])
        self.layer_idx = layer_idx

    def forward(self, permuted_local_hidden_states: torch.Tensor, tokens_per_expert: torch.Tensor):
        """Returns (output, output_bias); with `add_bias_linear` output_bias holds, row by row, the
        fc2 bias of the row's expert (mlp.py:200-207), which the dispatcher weights and combines
        like the output; with a single local expert it is that expert's [H] bias (mlp.py:184-186)."""
        if self.num_local_experts == 1:
            return self.local_experts[0](permuted_local_hidden_states)
        counts = tokens_per_expert.tolist()  # one host read, as in the reference (mlp.py:188)
        rows, total = permuted_local_hidden_states.shape[0], sum(counts)
        tokens_list = torch.split(permuted_local_hidden_states[:total], counts)
        outs, biases = [], []
        for expert, tokens in zip(self.local_experts, tokens_list):
            out, out_bias = expert(tokens)
            outs.append(out)
            if self.add_bias:
                biases.append(expand_bias(out_bias, tokens.shape[0]))
        if total < rows:  # the dispatcher sized the buffer by an upper bound: unused rows stay zero
            pad = permuted_local_hidden_states.new_zeros(rows - total, outs[0].shape[1])
            outs.append(pad)
            if self.add_bias:
                biases.append(pad)
        return torch.cat(outs, dim=0), (torch.cat(biases, dim=0) if self.add_bias else None)


class SharedExpertMLP(torch.nn.Module):
    """Dense gated MLP applied to every token (mlp.py:215-400), width
    `moe_shared_expert_intermediate_size`, with the reference's parameter names and layouts:
    `linear_fc1.weight [2Fs, H]` (gate rows first, then up rows), `linear_fc2.weight [H, Fs]`,
    `gate_weight [1, H]` when `gate` (output * sigmoid(x . gate_weight), mlp.py:271-278).

    With `config.moe_shared_expert_overlap` the reference's staged interface is available
    (pre_forward_comm, linear_fc1_forward_and_act, linear_fc2_forward, post_forward_comm,
    get_output): the stages enqueue on a stream of the class, so the dense products run beside
    the dispatch and the routed experts, and get_output makes the current stream wait for them.
    Where the layer's work is too little to pay for the second stream (`_stage_stream`), the stages
    enqueue on the current one."""

    stream = None  # shared by all instances, default priority
    overlap_min_us, overlap_min_us_captured = 150.0, 1.0  # see _stage_stream

    def __init__(self, config: MoEConfig, gate: bool = False, device=None):
        super().__init__()
        self.config = config
        assert config.add_bias_linear is False, "bias is not supported in the shared experts"
        assert config.gated_linear_unit, "the shared experts here are a gated (SwiGLU / GeGLU) MLP"
        self.act = _act_name(config)
        Fs = config.moe_shared_expert_intermediate_size
        assert Fs is not None
        device = torch.cuda.current_device() if device is None else device
        H = config.hidden_size
        self.linear_fc1 = _Linear(H, 2 * Fs, config, device)
        self.linear_fc2 = _Linear(Fs, H, config, device)
        self.use_shared_expert_gate = gate
        self.gate_weight = None
        if gate:
            self.gate_weight = Parameter(torch.empty(1, H, device=device, dtype=config.params_dtype))
            torch.nn.init.normal_(self.gate_weight, mean=0.0, std=config.init_method_std)
        self.overlap = bool(getattr(config, "moe_shared_expert_overlap", False))
        self._staged = {}
        if self.overlap and SharedExpertMLP.stream is None:
            SharedExpertMLP.stream = torch.cuda.Stream(device=device)

    # -- the three pieces of the forward ----------------------------------------------------------
    def _gate_score(self, x2d):
        from .router import _GateProjection  # the one-expert case of the gate projection kernels

        w = self.gate_weight if self.gate_weight.dtype == x2d.dtype else self.gate_weight.to(x2d.dtype)
        if not ops.gate_supported(x2d, w):
            raise ValueError("shared-expert gate: unsupported operands (dtype %s, hidden size %d)"
                             % (x2d.dtype, x2d.shape[-1]))
        logits = _GateProjection.apply(x2d, w, x2d.dtype)
        return torch.sigmoid(logits)

    def _fc1_act(self, x2d):
        # the SwiGLU input goes to the backward as fp8 where the reference's fused branch would
        # store it so (mlp.py:316-330: bias_activation_fusion, SiLU, activation_func_fp8_input_store)
        cfg = self.config
        fp8 = (getattr(cfg, "bias_activation_fusion", False) and self.act == "silu"
               and getattr(cfg, "activation_func_fp8_input_store", False))
        return glu(self.linear_fc1(x2d), self.act, fp8)

    def _finish(self, fc2_out, gate_score):
        if gate_score is None:
            return fc2_out
        from .moe_utils import scale_rows

        return scale_rows(fc2_out, gate_score)

    def forward(self, hidden_states: torch.Tensor) -> torch.Tensor:
        shape = hidden_states.shape
        x = hidden_states.reshape(-1, shape[-1]).contiguous()
        score = self._gate_score(x) if self.use_shared_expert_gate else None
        out = self._finish(self.linear_fc2(self._fc1_act(x)), score)
        return out.view(shape)

    # -- staged interface (mlp.py:280-400) ----------------------------------------------------------
    def _stage_stream(self, x):
        """The stream of the stages: the side stream or the current one.  The second stream costs the host 80 to 150 us
        in the forward and 80 in the backward (event records, stream switches, waits between the autograd
        nodes of two streams), and gains 1 to 19 % of the GPU's time.  So it takes a layer whose forward keeps the
        GPU busy beyond the launches' own time: its weights at 4.5 TB/s or its products at 800 TFLOP/s (fp32: 120),
        whichever is longer.  us per step with the side stream / without (estimate): 708 tokens of 192, 32 experts
        of 512, shared 4336 685 / 520 (5); 8345 of 1408, 8 of 384, top 4, shared 384 843 / 1005 (169); 512 of
        2048, 64 of 1408, top 6, shared 2816 977 / 999 (248); forward alone 512 of 1024, 16 of 2048, shared 4096 216
        / 162 (50); 16 of 2048, 64 of 1408, top 6, shared 2816 245 / 269 (248).
        A graph that is being captured costs the host nothing when it is replayed, so all but the smallest layers take the
        second stream there.  us of a replayed forward: 512 of 1024, 16 of 2048, shared 4096 125 / 136 (50); 4 of 512, 8 of
        1024, shared 1024 68 / 71 (6); 128 of 128, 4 of 256, shared 512 70 / 63 (0.3)."""
        cfg, H = self.config, x.shape[-1]
        tokens = x.numel() // H if H else 0
        experts, rows = cfg.num_moe_experts or 0, tokens * (cfg.moe_router_topk or 0)
        routed, shared = cfg.moe_ffn_hidden_size or 0, cfg.moe_shared_expert_intermediate_size
        weights = 3.0 * x.element_size() * H * (min(experts, rows) * routed + shared)
        products = 6.0 * H * (rows * routed + tokens * shared)
        us = max(weights / 4.5e6, products / (1.2e8 if x.dtype == torch.float32 else 8e8))
        least = self.overlap_min_us_captured if torch.cuda.is_current_stream_capturing() else self.overlap_min_us
        return SharedExpertMLP.stream if us >= least else torch.cuda.current_stream()

    def _stage(self):
        stream = self._staged["stream"]
        return contextlib.nullcontext() if stream == torch.cuda.current_stream() else torch.cuda.stream(stream)

    def pre_forward_comm(self, input):
        assert self.overlap, "stages out of order"
        # a forward that raised between two stages leaves its pieces behind: start afresh
        self._staged = {}
        stream, cur = self._stage_stream(input), torch.cuda.current_stream()
        if stream != cur:
            stream.wait_stream(cur)
        self._staged = {"shape": input.shape, "stream": stream}
        with self._stage():
            x = input.reshape(-1, input.shape[-1]).contiguous()
            if stream != cur:
                x.record_stream(stream)
            self._staged["x"] = x
            self._staged["score"] = self._gate_score(x) if self.use_shared_expert_gate else None

    def linear_fc1_forward_and_act(self, overlapped_comm_output=None):
        assert self.overlap and "x" in self._staged, "stages out of order"
        with self._stage():
            self._staged["act"] = self._fc1_act(self._staged.pop("x"))

    def linear_fc2_forward(self, overlapped_comm_output=None):
        assert self.overlap and "act" in self._staged, "stages out of order"
        with self._stage():
            self._staged["fc2"] = self.linear_fc2(self._staged.pop("act"))

    def post_forward_comm(self):
        assert self.overlap and "fc2" in self._staged, "stages out of order"  # no collective at TP 1

    def get_output(self):
        assert self.overlap and "fc2" in self._staged, "stages out of order"
        with self._stage():
            out = self._finish(self._staged["fc2"], self._staged["score"]).view(self._staged["shape"])
        stream, cur = self._staged["stream"], torch.cuda.current_stream()
        self._staged = {}
        if stream != cur:
            cur.wait_stream(stream)
            out.record_stream(cur)
        return out
