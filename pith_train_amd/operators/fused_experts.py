"""A whole SwiGLU expert block (fused gate_up projection -> SwiGLU -> down projection) as one
autograd node, for the FP8 path.

Composition and arithmetic are those of ``Qwen35MoeExperts.forward``
(models/qwen35_moe.py:190-200) built from ``FP8GroupedLinearFunc`` (grouped_linear.py:104-236) and
``silu_mul`` (silu_mul.py:93-143); the results are bit-identical to that composition.  Being one
node lets two intermediate bf16 tensors stay out of memory: the SwiGLU output ``h`` (forward) and
its gradient ``[dgate | dup]`` (backward) are produced inside the kernels that quantise them.
The token permutation can be folded in as well (``row_map``, see ``FP8GroupedLinearFunc``).
"""

from __future__ import annotations

import torch

from .. import _lib
from .deepgemm_quantize import FP8
from .grouped_linear import dgrad_operand


def _cdiv(a: int, b: int) -> int:
    return (a + b - 1) // b


def _last(offs):
    """Device pointer to the last entry of the inclusive group offsets (= the number of grouped rows)."""
    return None if offs is None or offs.numel() == 0 else offs.data_ptr() + 4 * (offs.numel() - 1)


def silu_mul_quant(gate_up: torch.Tensor, grouped_mm_offs: torch.Tensor | None = None):
    """``fp8cast_rowwise_colwise_t(silu_mul(gate_up[:, :I], gate_up[:, I:]))`` in one pass.  With
    ``grouped_mm_offs`` only the rows below its last entry are processed (the tensors may be sized
    for more rows than the routing produced)."""
    M, two_i = gate_up.shape
    half = two_i // 2
    dev = gate_up.device
    tok = torch.empty((M, half), dtype=FP8, device=dev)
    tok_s = torch.empty((M, _cdiv(half, 128)), dtype=torch.float32, device=dev)
    ch_t = torch.empty((half, M), dtype=FP8, device=dev)
    ch_s = torch.empty((M // 128, half), dtype=torch.float32, device=dev)
    _lib.call(
        "pt_silu_mul_quant_rowwise_colwise", gate_up.data_ptr(), M, half, gate_up.stride(0),
        tok.data_ptr(), tok_s.data_ptr(), ch_t.data_ptr(), ch_s.data_ptr(), _last(grouped_mm_offs),
        _lib.stream_ptr(dev),
    )  # fmt: skip
    return tok, tok_s, ch_t, ch_s


def silu_mul_bwd_quant(grad_h: torch.Tensor, gate_up: torch.Tensor, grouped_mm_offs: torch.Tensor | None = None):
    """``fp8cast_rowwise_colwise_t`` of the SwiGLU gradient ``[dgate | dup]`` in one pass (rows
    limited as in :func:`silu_mul_quant`)."""
    M, two_i = gate_up.shape
    half = two_i // 2
    dev = gate_up.device
    tok = torch.empty((M, two_i), dtype=FP8, device=dev)
    tok_s = torch.empty((M, _cdiv(two_i, 128)), dtype=torch.float32, device=dev)
    ch_t = torch.empty((two_i, M), dtype=FP8, device=dev)
    ch_s = torch.empty((M // 128, two_i), dtype=torch.float32, device=dev)
    _lib.call(
        "pt_silu_mul_bwd_quant_rowwise_colwise", grad_h.data_ptr(), grad_h.stride(0), gate_up.data_ptr(),
        gate_up.stride(0), M, half, tok.data_ptr(), tok_s.data_ptr(), ch_t.data_ptr(), ch_s.data_ptr(),
        _last(grouped_mm_offs), _lib.stream_ptr(dev),
    )  # fmt: skip
    return tok, tok_s, ch_t, ch_s


def clamped_swiglu_quant(gate_up: torch.Tensor, alpha: float, limit: float, grouped_mm_offs: torch.Tensor | None = None):
    """``fp8cast_rowwise_colwise_t(clamped_swiglu(gate_up, alpha, limit))`` in one pass (interleaved
    (gate, up) pairs, clamped_swiglu.py:95-155); rows limited as in :func:`silu_mul_quant`."""
    M, two_i = gate_up.shape
    half = two_i // 2
    dev = gate_up.device
    tok = torch.empty((M, half), dtype=FP8, device=dev)
    tok_s = torch.empty((M, _cdiv(half, 128)), dtype=torch.float32, device=dev)
    ch_t = torch.empty((half, M), dtype=FP8, device=dev)
    ch_s = torch.empty((M // 128, half), dtype=torch.float32, device=dev)
    _lib.call(
        "pt_clamped_swiglu_quant_rowwise_colwise", gate_up.data_ptr(), M, half, gate_up.stride(0), alpha, limit,
        tok.data_ptr(), tok_s.data_ptr(), ch_t.data_ptr(), ch_s.data_ptr(), _last(grouped_mm_offs),
        _lib.stream_ptr(dev),
    )  # fmt: skip
    return tok, tok_s, ch_t, ch_s


def clamped_swiglu_bwd_quant(grad_h: torch.Tensor, gate_up: torch.Tensor, alpha: float, limit: float,
                             grouped_mm_offs: torch.Tensor | None = None):
    """``fp8cast_rowwise_colwise_t`` of the clamped SwiGLU's input gradient in one pass, plus
    ``col_sum`` ``[M / 128, 2I]`` fp32: the column sums of every 128-row tile of that (bf16-rounded)
    gradient, from which the bias gradient of the projection before it is summed per group."""
    M, two_i = gate_up.shape
    half = two_i // 2
    dev = gate_up.device
    tok = torch.empty((M, two_i), dtype=FP8, device=dev)
    tok_s = torch.empty((M, _cdiv(two_i, 128)), dtype=torch.float32, device=dev)
    ch_t = torch.empty((two_i, M), dtype=FP8, device=dev)
    ch_s = torch.empty((M // 128, two_i), dtype=torch.float32, device=dev)
    col_sum = torch.empty((M // 128, two_i), dtype=torch.float32, device=dev)
    _lib.call(
        "pt_clamped_swiglu_bwd_quant_rowwise_colwise", grad_h.data_ptr(), grad_h.stride(0), gate_up.data_ptr(),
        gate_up.stride(0), M, half, alpha, limit, tok.data_ptr(), tok_s.data_ptr(), ch_t.data_ptr(), ch_s.data_ptr(),
        col_sum.data_ptr(), _last(grouped_mm_offs), _lib.stream_ptr(dev),
    )  # fmt: skip
    return tok, tok_s, ch_t, ch_s, col_sum


def supported(x: torch.Tensor, w_gate_up: torch.Tensor, w_down: torch.Tensor) -> bool:
    """bf16 activations, half width and hidden size multiples of 8 (16-byte accesses)."""
    gate_up, down = w_gate_up.shape, w_down.shape
    return x.dtype == torch.bfloat16 and gate_up[1] == 2 * down[2] and down[2] % 8 == 0 and down[1] % 8 == 0


def compose_row_maps(row_map: torch.Tensor, expand_idx: torch.Tensor, n_src: int) -> torch.Tensor:
    """``expand_idx[row_map]`` with the negative (padding) entries of ``row_map`` kept negative:
    the source row (among ``n_src``) of every grouped row when the routed rows are themselves an
    expansion (``expand_idx``) of deduplicated rows."""
    assert row_map.dtype == torch.int32 and expand_idx.dtype == torch.int64
    out = torch.empty_like(row_map)
    _lib.call(
        "pt_compose_row_map", row_map.contiguous().data_ptr(), row_map.numel(), expand_idx.contiguous().data_ptr(),
        expand_idx.numel(), n_src, out.data_ptr(), _lib.stream_ptr(row_map.device),
    )  # fmt: skip
    return out


FEW_ROWS = 64  # group alignment of forwards that no backward follows, see few_rows_per_expert


def few_rows_per_expert(rows: int, num_groups: int) -> bool:
    """Whether a forward without a backward pads its groups to 64 rows instead of 128 and takes the GEMM tiles
    of that height.  Such a forward reads every expert's weights for a handful of rows, and half of a
    128-row tile would be padding; with more rows than this most groups need a second 64-row tile,
    which reads the weight panel again.  Expert blocks (2048 x 768 x 128, 2048 x 1408 x 64 and 2880 x 2880 x 32
    hidden x width x experts, equal popularity), us with 64 / 128 rows: 16 rows an expert 163 / 211, 143 / 174,
    221 / 261; 48 178 / 217, 151 / 178, 224 / 264; 64 208 / 220, 175 / 181, 273 / 263; 80 237 / 225, 200 / 184,
    301 / 273.  With Zipf-distributed popularity the gain ends between 40 and 80."""
    return rows <= 48 * num_groups


def _prepare(x, grouped_mm_offs, row_map, expand_idx, scatter):
    """The checked ``(row_map, expand_idx, scatter)`` of a block on ``x`` (a ``[T, k, K]`` view of one row per
    token counts as its T * k rows)."""
    _lib.require_cuda(x)
    # three dimensions: one row per token, seen k times
    assert x.dim() == 2 or (x.dim() == 3 and row_map is not None and expand_idx is None and (x.stride(1) == 0 or x.shape[1] == 1)), (
        f"expected [rows, width] or an expanded [tokens, k, width] view, got {tuple(x.shape)} with strides {x.stride()}")
    assert expand_idx is None or row_map is not None, "expand_idx needs the row map of the scatter"
    if row_map is not None:
        assert row_map.dtype == torch.int32 and row_map.shape[0] % 128 == 0
        row_map = row_map.contiguous()
    else:
        assert x.dim() == 2 and x.shape[0] % 128 == 0, f"grouped rows must be a multiple of 128, got {x.shape[0]}"
    if expand_idx is not None:
        assert expand_idx.dtype == torch.int64
        expand_idx = expand_idx.contiguous()
    return row_map, expand_idx, scatter and row_map is not None


def _check_biases(x, w_down, biases):
    """The GEMM stores add a row of the bias per group, addressed by the weights' sizes."""
    G, H, half = w_down.shape
    for bias, width in zip(biases, (2 * half, H)):
        assert bias is None or (bias.shape == (G, width) and bias.dtype == x.dtype), (
            f"bias must be {x.dtype} {(G, width)}, got {bias.dtype} {tuple(bias.shape)}")


def _node(x, w_gate, w_up, w_down, grouped_mm_offs, q_gate_up, q_down, row_map, expand_idx=None, scatter=True, clamp=None, biases=(None, None)):
    """The autograd node of the three functions below (``csrc/host.cpp``): the forward is one library call that
    queues every launch of it, and so is the backward but for its input gradient.  ``w_gate`` and
    ``w_up`` are the parameters whose gradients the gate_up weight gradient is written to; without
    ``w_up`` the former is the fused ``[G, 2I, K]`` one.  ``expand_idx`` (with
    ``row_map``): ``x`` holds deduplicated rows and routed row i is ``x[expand_idx[i]]``; the result
    has one row per routed row, and the backward sums the gradients of the rows that share a source
    row.  ``scatter`` (with ``row_map``): the result comes back un-permuted.  ``clamp``: ``(alpha,
    limit)`` of the clamped SwiGLU, whose projections have the two ``biases``.  ``x`` may be an expanded
    ``[T, k, K]`` view of one row per token (routed row i is token i // k).  The weight gradients go to
    ``.grad``, or to the ``WeightGradStore`` queue."""
    row_map, expand_idx, scatter = _prepare(x, grouped_mm_offs, row_map, expand_idx, scatter)
    if biases != (None, None):
        _check_biases(x, w_down, biases)
    M = x.shape[0] if row_map is None else row_map.shape[0]
    weights = w_gate if w_up is None else (w_gate, w_up)
    return _lib.host().experts(
        x, w_gate, w_up, w_down, *biases, grouped_mm_offs, q_gate_up[:2], q_down[:2], dgrad_operand(q_gate_up, weights, M),
        dgrad_operand(q_down, w_down, M), row_map, expand_idx, scatter, clamp, _lib.stream_ptr(x.device),
    )  # fmt: skip


def wants_backward(x: torch.Tensor, *weights: torch.Tensor) -> bool:
    """Whether a backward can follow a forward on these tensors."""
    return torch.is_grad_enabled() and (x.requires_grad or any(w.requires_grad for w in weights))


def forward_only(x, w_down, grouped_mm_offs, q_gate_up, q_down, row_map=None, expand_idx=None, scatter=True,
                 clamp=None, biases=(None, None), few_rows=False):
    """The forward of the nodes below when no backward follows: nothing is kept, the quantisers leave out
    the transposed operands of the weight gradients, and the groups may be multiples of 64 rows
    (``few_rows``)."""
    row_map, expand_idx, scatter = _prepare(x, grouped_mm_offs, row_map, expand_idx, scatter)
    repeat = 1
    if x.dim() == 3:
        repeat, x = x.shape[1], x[:, 0]
    if x.stride(1) != 1:
        x = x.contiguous()
    _check_biases(x, w_down, biases)
    if biases[0] is not None:
        biases = [b.detach().contiguous() for b in biases]
    return _lib.host().experts_forward(
        x, repeat, row_map, expand_idx, grouped_mm_offs, *q_gate_up[:2], *q_down[:2], w_down.shape[2], *biases, scatter, clamp is not None,
        *(clamp or (0.0, 0.0)), False, few_rows, _lib.stream_ptr(x.device),
    )[0]  # fmt: skip


class FP8SwiGLUExpertsFunc:
    @staticmethod
    def apply(x, w_gate_up, w_down, grouped_mm_offs, ks, ks_tensor, q_gate_up, q_down, row_map=None, expand_idx=None):
        """``x`` is ``[M, K]`` grouped rows, or with ``row_map`` (int32 ``[M]``) the un-permuted
        ``[m, K]`` tokens; the result has the same row layout as ``x``.  ``row_map`` may be longer
        than the grouped rows (its tail negative): every kernel takes the real row count from
        ``grouped_mm_offs`` on the device, so no host-side size is needed (``ks`` may be None)."""
        return _node(x, w_gate_up, None, w_down, grouped_mm_offs, q_gate_up, q_down, row_map, expand_idx)


class FP8SwiGLUSplitExpertsFunc:
    """The same node for experts that keep gate and up as separate parameters
    (``Qwen3MoeExperts`` / ``DeepSeekV2Experts``, models/qwen3_moe.py:45-65): ``q_gate_up`` is the
    two weights quantised into one fused operand (:func:`fp8cast_blockwise_transpose_batched_cat`),
    so the tokens are quantised once and one GEMM each way serves both projections; the weight
    gradients are written to the two parameters separately."""

    @staticmethod
    def apply(x, w_gate, w_up, w_down, grouped_mm_offs, q_gate_up, q_down, row_map=None, expand_idx=None):
        return _node(x, w_gate, w_up, w_down, grouped_mm_offs, q_gate_up, q_down, row_map, expand_idx)


def supported_split(x: torch.Tensor, w_gate: torch.Tensor, w_up: torch.Tensor, w_down: torch.Tensor) -> bool:
    """As :func:`supported`, and the halves must be whole 128-row blocks of the fused operand."""
    gate, down = w_gate.shape, w_down.shape
    return x.dtype == torch.bfloat16 and gate[1] == down[2] and gate[1] % 128 == 0 and down[1] % 8 == 0 and gate == w_up.shape


class FP8ClampedSwiGLUExpertsFunc:
    """The GPT-OSS expert block (models/gpt_oss.py:139-157: gate_up projection + bias, clamped
    SwiGLU on interleaved pairs, down projection + bias) as one node.  Outputs, input gradient,
    weight gradients and the down bias gradient have the bits of the composition of
    ``FP8GroupedLinearFunc`` (biases in the GEMM stores) and ``clamped_swiglu``; the activation
    and its gradient are never written as bf16 tensors, and the gate_up bias gradient is summed
    from per-tile column sums that the backward's quantisation produces (fp32, another order of
    additions than the segmented sum over the materialised gradient: same value up to fp32
    rounding before the cast to the bias dtype).

    ``row_map`` (int32 ``[M]``, from the scatter): ``x`` is the un-permuted ``[m, K]`` token tensor;
    with ``scatter_output`` the result comes back un-permuted as well."""

    @staticmethod
    def apply(x, w_gate_up, b_gate_up, w_down, b_down, grouped_mm_offs, q_gate_up, q_down, alpha, limit,
                row_map=None, scatter_output=False):
        assert not scatter_output or row_map is not None, "scatter_output needs the row map"
        return _node(x, w_gate_up, None, w_down, grouped_mm_offs, q_gate_up, q_down, row_map, None, scatter_output,
                     (float(alpha), float(limit)), (b_gate_up, b_down))
