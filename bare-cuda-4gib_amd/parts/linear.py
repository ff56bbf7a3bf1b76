"""y = x W^T for a weight stored [out, in] (the orientation a checkpoint stores
a linear layer in; reference: engine/include/llm/kernels.h:48-57), and the
choice of kernel for it (reference: matmul dispatch, engine/src/model.cpp:153-192):
up to 64 rows the weight-streaming kernel (with RMSNorm fused in up to 16 rows),
beyond that the tiled matrix-core kernel, and the plain float kernel for
what those refuse (k no multiple of 8).  Float32 operands go to the
float32 matrix-core kernel where it takes them (which up to 64 rows prepares and
finishes norms too), else to the plain one."""
from __future__ import annotations

from typing import Optional, Union

import torch

from ..csrc import ops
from .lazy import Normed


def _fused_norm(x: Normed, w, epilogue: int) -> Optional[torch.Tensor]:
    if x._tensor is not None:
        return None
    scale = x.fusable_scale()
    if scale is None or not ops.gemm_normed_supported(x.x, x.n_rows, scale[0], w):
        return None
    return ops.gemm_normed(x.x, x.rows, x.n_rows, scale[0], scale[1], w, epilogue)


def absorbs_norm(norm, w, n_rows: int) -> bool:
    """Whether a product of n_rows rows of the stream with this weight absorbs the norm before it (_fused_norm)."""
    scale = norm.fusable() if hasattr(norm, "fusable") else None
    return scale is not None and ops.absorbs_norm(n_rows, scale[0], w)


def _prepare(x: Normed, w) -> None:
    """What the product would make of the norm in each of its workgroups, by a kernel before it where that is the faster way (the same bits)."""
    if x.n_rows > ops.NORMED_MAX_ROWS or x.pre is not None or x._tensor is not None or not ops.norm_apart(x.n_rows, w):
        return
    scale = x.fusable_scale()
    if scale is not None and ops.gemm_normed_supported(x.x, x.n_rows, scale[0], w):
        x.pre = ops.rmsnorm_prepare(x.x, x.rows, x.n_rows, *scale)


def _prepared_norm(x: Normed, w, epilogue: int) -> Optional[torch.Tensor]:
    """The product from what the product before left for this norm, or a kernel before it makes, where there is such a thing."""
    _prepare(x, w)
    if x.pre is None or x._tensor is not None:
        return None
    if x.pre.xb.dtype == torch.float32:
        act = {ops.EPI_STORE_F32: None, ops.EPI_SWIGLU: "silu", ops.EPI_GEGLU: "gelu_tanh"}.get(epilogue, "")
        return ops.gemm_f32_prenormed(x.pre, w, act) if act != "" else None
    if not ops.gemm_prenormed_supported(x.pre, w, epilogue):
        return None
    return ops.gemm_prenormed(x.pre, w, epilogue)


def linear(x: Union[torch.Tensor, Normed], w, out_dtype: Optional[torch.dtype] = None,
           accumulate_into: Optional[torch.Tensor] = None, ctx=None, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x [M, K] times w [N, K] transposed (w a tensor or an ops.StreamedWeight).  With
    ``accumulate_into`` (the float32 residual stream) the product is added to it in place; with
    ``ctx`` too, and a norm named as the next reader of the stream (``ctx.handoff.reading_next``), the
    product prepares that norm where its kernel can and leaves the result with the handoff: the norm
    itself (ops.Finished) where the product cuts k over workgroups anyway -- the kernel that adds the parts
    up norms the stream on its way, which serves every reader -- or else, if the reader takes that, the parts
    of the norm that a product can finish (ops.Prenormed).  ``bias`` (float32, a number a column): added to every row
    with an adding product, in whichever kernel adds it."""
    if isinstance(accumulate_into, ops.Fresh):        # nothing to add to yet: the product itself, in float32
        if accumulate_into.tensor is None and bias is not None:
            accumulate_into.tensor = torch.zeros((x.shape[0], w.shape[0]), dtype=torch.float32, device=x.device)
        if accumulate_into.tensor is not None:
            return linear(x, w, accumulate_into=accumulate_into.tensor, ctx=ctx, bias=bias)
        accumulate_into.tensor = linear(x, w, out_dtype=torch.float32)
        return accumulate_into.tensor
    if isinstance(x, Normed):
        if accumulate_into is None and out_dtype in (torch.bfloat16, torch.float32):
            epi = ops.EPI_STORE_BF16 if out_dtype == torch.bfloat16 else ops.EPI_STORE_F32
            fused = _prepared_norm(x, w, epi)
            if fused is None:
                fused = _fused_norm(x, w, epi)
            if fused is not None:
                return fused
        x = x.tensor()
    reading = ctx.handoff.reading_next if ctx is not None and accumulate_into is not None else None
    if reading is not None:
        norm, takes_parts = reading
        scale = norm.fusable() if hasattr(norm, "fusable") else None
        if scale is not None and ops.gemm_parts_supported(x, w, accumulate_into, scale[0]):
            ctx.handoff.leave(norm, ops.gemm_parts_accumulate_norm(x, w, accumulate_into, scale[0], scale[1], checked=True, bias=bias))
            return accumulate_into
        if scale is not None and takes_parts and ops.gemm_emit_supported(x, w, accumulate_into, scale[0]):
            ctx.handoff.leave(norm, ops.gemm_accumulate_emit(x, w, accumulate_into, scale[0], scale[1], bias=bias))
            return accumulate_into
        left = ops.gemm_f32_emit(x, w, accumulate_into, scale[0], scale[1], bias=bias) if scale is not None and takes_parts else None
        if left is not None:
            ctx.handoff.leave(norm, left)
            return accumulate_into
    fast = ops.gemm_fast(x, w, out_dtype, accumulate_into, bias=bias)
    if fast is None and out_dtype in (None, torch.float32):
        fast = ops.gemm_f32(x, w, accumulate_into, bias=bias)
    if fast is not None:
        return fast
    return ops.gemm_generic(x, w, out_dtype, accumulate_into, bias=bias)


def linear_squared_relu(x: Union[torch.Tensor, Normed], w, out_dtype: torch.dtype) -> torch.Tensor:
    """max(x W^T, 0)^2: applied to the float sums inside the product's kernel where a matrix-core kernel takes the
    operands (with the norm fused or prepared like any product's), else by a kernel behind it."""
    if isinstance(x, Normed):
        if out_dtype == torch.bfloat16:
            fused = _prepared_norm(x, w, ops.EPI_SQUARED_RELU)
            if fused is None:
                fused = _fused_norm(x, w, ops.EPI_SQUARED_RELU)
            if fused is not None:
                return fused
        x = x.tensor()
    fast = ops.gemm_fast(x, w, out_dtype, squared_relu=True)
    if fast is not None:
        return fast
    z = linear(x, w, out_dtype=out_dtype)
    return ops.squared_relu(z, out=z)


def linear_xielu(x: Union[torch.Tensor, Normed], w, pq: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    """xielu(x W^T) with its two numbers pq: inside the product's kernel where few rows stream the weights (with the norm prepared, if
    it was), else by a kernel behind it."""
    if out_dtype == torch.bfloat16:
        if isinstance(x, Normed):
            _prepare(x, w)
            if x.pre is not None and x._tensor is None:
                fast = ops.gemm_xielu(x.pre.xb, w, pq, pre=x.pre)
                if fast is not None:
                    return fast
            z = _fused_norm(x, w, ops.EPI_STORE_BF16)
            if z is not None:
                return ops.xielu(z, pq, out=z)
            x = x.tensor()
        fast = ops.gemm_xielu(x, w, pq)
        if fast is not None:
            return fast
    z = linear(x, w, out_dtype=out_dtype)
    return ops.xielu(z, pq, out=z)


def linear_swiglu(x: Union[torch.Tensor, Normed], w_gate_up, interleaved: bool = False, act: str = "silu") -> torch.Tensor:
    """act(x Wg^T) * (x Wu^T) (``act``: "silu", or "gelu_tanh", the gelu written with tanh) for w_gate_up = gate rows followed by up rows, or (interleaved)
    blocks of eight gate rows and the eight up rows of the same outputs."""
    if isinstance(x, Normed):
        fused = None
        if interleaved and w_gate_up.shape[0] % 16 == 0:
            fused = _prepared_norm(x, w_gate_up, ops.gated_epilogue(act))
            if fused is None:
                fused = _fused_norm(x, w_gate_up, ops.gated_epilogue(act))
        elif not interleaved and x.pre is not None and x.pre.xb.dtype == torch.float32:
            fused = _prepared_norm(x, w_gate_up, ops.gated_epilogue(act))
        if fused is not None:
            return fused
        x = x.tensor()
    return ops.gemm_swiglu(x, w_gate_up, interleaved, act)
