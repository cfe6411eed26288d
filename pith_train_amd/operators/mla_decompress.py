"""FP8 decompression of the MLA latent through ``kv_b`` - the local step inside the ring of the
reference's MLA ring attention, on the dense FP8 kernels of this library.

``mla_decompress`` is ``_mla_decompress`` of the reference (operators/ring_attention.py:428-457):
the latent block is quantised row-wise here (it differs every ring hop) and multiplied with the
``kv_b`` weight the caller quantised once per micro-batch.  ``mla_decompress_backward`` is the
FP8 branch of the ring's backward (operators/ring_attention.py:636-652): the latent block is
re-quantised for the weight gradient instead of being kept from the forward, and both gradients
come back in fp32.  The ring itself (send/receive of latent blocks, flash attention calls, the
online-softmax merge) is not part of this library.
"""

from __future__ import annotations

from typing import Optional, Tuple

import torch
import torch.nn.functional as F

from .deepgemm_quantize import fp8cast_rowwise_blockwise_transpose
from .linear import fp8_act_weight_gemm, fp8_act_weight_gemm_heads, fp8_dgrad_wgrad, fp8_dgrad_wgrad_heads


def mla_decompress(
    normed_kv: torch.Tensor,
    kv_b_weight: torch.Tensor,
    num_heads: int,
    qk_nope_head_dim: int,
    v_head_dim: int,
    *,
    use_fp8: bool = False,
    weight_fp8: Optional[torch.Tensor] = None,
    scale_weight: Optional[torch.Tensor] = None,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Latent block ``[b, n, lora_rank]`` -> per-head ``(k_nope [b, n, heads, qk_nope], value
    [b, n, heads, v] contiguous)`` via ``y = x @ kv_b.T``."""
    b, n, _ = normed_kv.shape
    if use_fp8:
        x2d = normed_kv.reshape(b * n, normed_kv.shape[-1])
        # the GEMM stores both parts where they belong (4096 rows: the copy of the values took 10 us)
        parts = fp8_act_weight_gemm_heads(x2d, weight_fp8, scale_weight, num_heads, qk_nope_head_dim, v_head_dim)
        if parts is not None:
            return parts[0].view(b, n, num_heads, qk_nope_head_dim), parts[1].view(b, n, num_heads, v_head_dim)
        kv2d, _, _ = fp8_act_weight_gemm(x2d, weight_fp8, scale_weight)
        kv = kv2d.view(b, n, num_heads, qk_nope_head_dim + v_head_dim)
    else:
        kv = F.linear(normed_kv, kv_b_weight).view(b, n, num_heads, qk_nope_head_dim + v_head_dim)
    k_nope, value = torch.split(kv, [qk_nope_head_dim, v_head_dim], dim=-1)
    # value feeds the attention kernel, which wants it contiguous; k_nope is concatenated with the
    # rotary part by the caller, which copies it anyway
    return k_nope, value.contiguous()


def mla_decompress_backward(
    dk_nope: torch.Tensor,
    dvalue: torch.Tensor,
    nkv_blk: torch.Tensor,
    weight_t_fp8: torch.Tensor,
    scale_weight_t: torch.Tensor,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """``(dk_nope [b, n, heads, qk_nope], dvalue [b, n, heads, v])`` and the hop's latent block
    ``nkv_blk [b, n, lora_rank]`` -> ``(d_nkv_blk [b, n, lora_rank] fp32, dW_blk [out, lora_rank]
    fp32)`` through the FP8 dgrad / wgrad of the dense linear."""
    b, n, lora_rank = nkv_blk.shape
    out_features = dk_nope.shape[2] * (dk_nope.shape[3] + dvalue.shape[3])
    # the quantiser reads both parts in place and the GEMMs store fp32 (4096 rows: concatenation and casts took 37 us)
    grads = fp8_dgrad_wgrad_heads(dk_nope.flatten(0, 1), dvalue.flatten(0, 1), weight_t_fp8, scale_weight_t,
                                  nkv_blk.reshape(b * n, lora_rank), lora_rank)  # fmt: skip
    if grads is not None:
        return grads[0].view(b, n, lora_rank), grads[1]
    dy2d = torch.cat([dk_nope, dvalue], dim=-1).reshape(b * n, out_features).to(nkv_blk.dtype)
    _, _, x_t_fp8, scale_x_t = fp8cast_rowwise_blockwise_transpose(nkv_blk.reshape(b * n, lora_rank), _padded=True)
    d_nkv_2d, dW_blk = fp8_dgrad_wgrad(dy2d, weight_t_fp8, scale_weight_t, x_t_fp8, scale_x_t, lora_rank, _zero_padded=True)
    return d_nkv_2d.view(b, n, lora_rank).to(torch.float32), dW_blk.to(torch.float32)
