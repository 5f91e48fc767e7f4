"""Matrix products of the parts: out (=|+=) a @ weight.T with weights [out_features, in_features]
as checkpoints store them (no bias).  The kernel is chosen by the operands' storage: 32-bit
operands take the exact kernel; bfloat16 operands take the matrix-core kernels where their
shape rules allow and the exact kernel otherwise.  `a` may be a norm not yet applied
(`NormedRows`); it is applied here, by the norm's own kernel (which also gathers the rows it names).
Applying it inside the product's kernel was measured and did not pay: as a prologue it costs what the
separate kernel costs, and commuted into the epilogue with the product reading the 32-bit rows it
makes the product's loop twice as slow.  What pays, for a few rows, is to split it over the two
products around it (`HandedRows`, `linear_onto`): the one that writes the rows also writes them
times the norm's weights in bfloat16 and the pieces of their sums of squares, the one that reads them
multiplies its results by the rows' rsqrt(mean square + eps)."""
from __future__ import annotations

import torch

from ..kernels import ops
from .norm import HandedRows, NormedRows, NormToMake, ReadyRows


def linear(a, weight: torch.Tensor, out: torch.Tensor, accumulate: bool = False, gated: bool = False, gate_limit: float = 0.0,
           ctx=None) -> torch.Tensor:
    """gated: weight is [gate; up] interleaved by `ops.interleave_gate_up` and out = act(gate) * up (bfloat16 only); True or "silu"
    for SiLU, "gelu_tanh" for the tanh form of GELU, "swish_clamped" (with `gate_limit`) for the clamped form.  ctx: the step the product is one
    of, whose counters (`ops.step_counters`) save it a launch where it has a use for them."""
    if isinstance(a, HandedRows):
        if (weight.dtype == torch.bfloat16 and ops.gemm_bf16_supports(a.scaled, weight, out)
                and ops.gemm_bf16_takes_norm(a.scaled.shape[0], weight.shape[0], weight.shape[1], gated)):
            return ops.gemm_bf16(a.scaled, weight, out, accumulate, gated, checked=True, norm_in=(a.squares, a.eps), gate_limit=gate_limit, ctx=ctx)
    if isinstance(a, NormedRows):
        a = a.materialize()
    if a.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and ops.gemm_bf16_supports(a, weight, out):
        return ops.gemm_bf16(a, weight, out, accumulate, gated, checked=True, gate_limit=gate_limit, ctx=ctx)
    if gated:
        raise ops.KernelError("the gated product exists for bfloat16 operands only")
    return ops.gemm_exact(a, weight, out, accumulate)


def linear_xielu(a, weight: torch.Tensor, params: torch.Tensor, columns: int, dtype: torch.dtype, out: torch.Tensor = None, into: torch.Tensor = None):
    """The product of `linear` with the activation of a feed-forward that has no gate in its epilogue, where a kernel does both
    (`ops.gemm_bf16_xielu`): its last `columns` columns come back activated, as `dtype` (in `into`, if given), the ones before go to out.  None where no
    kernel does, and out is as it was."""
    n, k = weight.shape
    rows = a.n_rows if isinstance(a, NormedRows) else a.shape[0]
    if not (weight.dtype == dtype == torch.bfloat16 and ops.gemm_bf16_xielu_takes(rows, n, k, n - columns)):
        return None
    norm_in = None
    if isinstance(a, HandedRows):
        if not (rows <= 16 and takes_handed_norm(weight, rows)):
            return None
        a, norm_in = a.scaled, (a.squares, a.eps)
    elif isinstance(a, NormedRows):
        a = a.materialize()                      # (kept by `a` for whoever asks next)
    if not ops.gemm_bf16_supports(a, weight, weight):
        return None
    mid = into if into is not None else torch.empty((rows, columns), dtype=dtype, device=weight.device)
    return ops.gemm_bf16_xielu(a, weight, params, mid, out, norm_in)


def linear_onto(a: torch.Tensor, weight: torch.Tensor, residual: torch.Tensor, then=None, ctx=None):
    """residual += a @ weight.T.  `then`: the norm that reads `residual` next, if it and its reader can take it half applied
    (see `HandedRows`); the product then also does the norm's share and the `HandedRows` are returned, None otherwise.  Or that norm as a
    `NormToMake`, for a reader that takes no other than a whole one: the rows come back normed where the product's kernel can."""
    if isinstance(then, NormToMake):
        norm, n, k = then.norm, weight.shape[0], weight.shape[1]
        if (a.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and residual.dtype == torch.float32 and ops.gemm_bf16_onto_norm_takes(residual.shape[0], n, k)
                and residual.stride(0) % 4 == 0 and residual.data_ptr() % 16 == 0 and norm.handed_weight().data_ptr() % 16 == 0 and ops.gemm_bf16_supports(a, weight, residual)):
            normed = torch.empty(residual.shape, dtype=torch.bfloat16, device=residual.device)
            return ReadyRows(norm, residual, ops.gemm_bf16_onto_norm(a, weight, residual, norm.handed_weight(), norm.eps, normed, checked=True))
        then = None
    if (then is not None and a.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and residual.dtype == torch.float32
            and residual.is_contiguous() and ops.gemm_bf16_supports(a, weight, residual)):
        rows, width = residual.shape
        parts = ops.gemm_bf16_norm_parts(rows, weight.shape[0], weight.shape[1])
        if parts:
            scaled = torch.empty((rows, width), dtype=torch.bfloat16, device=residual.device)
            squares = torch.empty((rows, parts), dtype=torch.float32, device=residual.device)
            ops.gemm_bf16(a, weight, residual, accumulate=True, checked=True, norm_out=(then.handed_weight(), scaled, squares), ctx=ctx)
            return HandedRows(then, residual, scaled, squares)
    linear(a, weight, residual, accumulate=True, ctx=ctx)
    return None


def takes_handed_norm(weight: torch.Tensor, n_rows: int, gated: bool = False) -> bool:
    """Whether `linear(handed rows, weight, ...)` finishes a norm handed on at this number of rows, rather than asking for the rows
    normed the ordinary way: exactly `linear`'s own conditions, for parts that must know beforehand (a part that reads normed
    rows after another part has changed the rows they were made of cannot fall back on them)."""
    n, k = weight.shape
    return (weight.dtype == torch.bfloat16 and k % 8 == 0 and weight.stride(1) == 1 and weight.stride(0) % 8 == 0 and weight.data_ptr() % 16 == 0
            and ops.gemm_bf16_takes_norm(n_rows, n, k, gated))


def activation_dtype_for(weight: torch.Tensor, compute_dtype: torch.dtype) -> torch.dtype:
    """What the input of a product with `weight` is stored as: bfloat16 only if both the compute
    dtype and the weight are; a weight kept in 32-bit gets 32-bit activations."""
    return torch.bfloat16 if compute_dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 else torch.float32
