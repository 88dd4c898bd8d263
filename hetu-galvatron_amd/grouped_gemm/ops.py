"""`grouped_gemm.ops.gmm`: differentiable grouped GEMM (call sites moe/mlp.py:106-112).

out[rows_e] = a[rows_e] @ op(b[e]); dA is the same product against the transposed weights,
dB[e] = a[rows_e]^T @ grad[rows_e] (zeros for an expert without rows)."""
from .. import _C
from .. import ops as _ops


def gmm(a, b, batch_sizes, trans_b=False):
    offsets = _ops.expert_offsets_from_batch_sizes(batch_sizes, a.device)
    return _C.host().grouped_gemm(a, b, offsets, trans_b)
