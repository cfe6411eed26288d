"""Top-k weighted combine of the expert outputs with the residual stream.

The memory-bound step right after the expert path: the single-rank branch of ``forward_stage5``
(models/qwen3_moe.py:229-237, and the same expression in the other model files)

    weighted = moe_outs.view(*topk_weight.shape, -1) * topk_weight.unsqueeze(-1)
    return residual + weighted.sum(dim=1).to(moe_outs.dtype).view(*residual.shape)

as one kernel each way instead of a product tensor, a reduction, a cast and an addition, and the
expert-parallel branch (models/qwen3_moe.py:238-245)

    permuted_probs = topk_weight.view(-1)[moe_local_idxs]
    token_indices = moe_local_idxs // topk_weight.shape[1]
    weighted = (moe_outs.float() * permuted_probs.unsqueeze(-1)).to(moe_outs.dtype)
    aggregated = moe_outs.new_zeros(topk_weight.shape[0], moe_outs.shape[-1])
    aggregated.scatter_add_(0, token_indices[:, None].expand_as(weighted), weighted)
    return residual + aggregated.view(*residual.shape)

likewise (:func:`moe_combine_ep`), with the order of the adds fixed: ascending row per token.
"""

from __future__ import annotations

import torch
from torch.autograd import forward_ad

from .. import _lib


def moe_combine(moe_outs: torch.Tensor, topk_weight: torch.Tensor, residual: torch.Tensor | None = None) -> torch.Tensor:
    """``residual + (moe_outs.view(T, k, H) * topk_weight[..., None]).sum(1).to(moe_outs.dtype)``.

    ``moe_outs`` is ``[T*k, H]`` (row ``t*k + j`` = expert output of token t's j-th choice),
    ``topk_weight`` float32 ``[T, k]``, ``residual`` any shape with ``T*H`` elements; the result
    has the residual's shape and ``moe_outs``' dtype.  Without a residual the result is the
    rounded weighted sum ``[T, H]`` itself (the last line of the models' ``reference_forward``,
    models/qwen3_moe.py:119)."""
    _lib.require_cuda(moe_outs, topk_weight, residual)
    assert moe_outs.ndim == 2 and topk_weight.ndim == 2, "moe_outs must be [T*k, H], topk_weight [T, k]"
    T, k = topk_weight.shape
    assert moe_outs.shape[0] == T * k, f"moe_outs has {moe_outs.shape[0]} rows, expected {T * k}"
    assert topk_weight.dtype == torch.float32, "topk_weight must be float32 (softmax scores)"
    assert residual is None or (residual.numel() == T * moe_outs.shape[1] and residual.dtype == moe_outs.dtype), (
        "residual must be [T, H] in moe_outs' dtype")
    return _lib.host().combine(moe_outs, topk_weight, residual, _lib.stream_ptr(moe_outs.device))


def moe_combine_ep(moe_outs: torch.Tensor, moe_local_idxs: torch.Tensor, topk_weight: torch.Tensor,
                   residual: torch.Tensor) -> torch.Tensor:
    """Expert-parallel combine: row r of ``moe_outs`` ``[R, H]`` is the expert output of the flat
    top-k slot ``moe_local_idxs[r]`` (token ``moe_local_idxs[r] // k``); entries are distinct (the
    dispatch sort's permutation, ep_dispatch.py:669-676).  Every row is weighted in fp32 and
    rounded, a token's rows are added in ascending r with every partial sum rounded to the
    storage type (a sequential ``scatter_add_``), and the residual is added last."""
    _lib.require_cuda(moe_outs, moe_local_idxs, topk_weight, residual)
    assert moe_outs.ndim == 2 and topk_weight.ndim == 2, "moe_outs must be [R, H], topk_weight [T, k]"
    T, k = topk_weight.shape
    R, H = moe_outs.shape
    assert moe_local_idxs.shape == (R,) and moe_local_idxs.dtype == torch.int64, "moe_local_idxs must be int64 [R]"
    assert R <= T * k, f"{R} rows for {T * k} top-k slots"
    assert residual.numel() == T * H and residual.dtype == moe_outs.dtype, "residual must be [T, H] in moe_outs' dtype"
    assert topk_weight.dtype == torch.float32, "topk_weight must be float32 (softmax scores)"
    return _lib.host().combine_ep(moe_outs, moe_local_idxs, topk_weight, residual, _lib.stream_ptr(moe_outs.device))


def token_branches(x: torch.Tensor, k: int, n: int):
    """``x`` ``[T, H]`` for a MoE block's branches: the expanded view ``[T, k, H]`` with one row per (token,
    choice) for the experts, and ``n`` (up to 3) times ``x`` itself.  The backward adds the branches'
    gradients, the k rows of the experts' included, in one pass with one rounding, where a reduction and an
    addition per branch would each read and write the whole tensor."""
    plain = not (torch.is_grad_enabled() and x.requires_grad) or torch.compiler.is_compiling() or torch._C._functorch.is_functorch_wrapped_tensor(x)
    if plain or forward_ad.unpack_dual(x).tangent is not None:
        return (x.unsqueeze(1).expand(-1, k, -1), *([x] * n))
    return _lib.host().branches(x, k, n, _lib.stream_ptr(x.device))
