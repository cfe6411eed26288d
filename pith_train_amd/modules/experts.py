"""Expert blocks of the supported model families and the stage-3 composition around them.

Mirrors the expert path of the reference's model files:
  * ``Qwen3MoeExperts``      - models/qwen3_moe.py:45-65   (gate, up, down as three grouped linears)
  * ``DeepSeekV2Experts``    - models/deepseek_v2.py:111-129
  * ``DeepSeekV2MLP``        - models/deepseek_v2.py:94-108 (dense shared expert)
  * ``Qwen35MoeExperts``     - models/qwen35_moe.py:179-200 (fused gate_up, concatenated halves)
  * ``GptOssExperts``        - models/gpt_oss.py:95-157     (fused interleaved gate_up, biases,
                                                              clamped SwiGLU)
  * ``forward_stage3``       - models/qwen3_moe.py:216-227  (expand -> scatter -> experts -> gather)

The constructors take plain sizes instead of Hugging Face config objects; everything else
(parameter names, shapes, call signatures) follows the reference so that checkpoints and callers
line up.
"""

from __future__ import annotations

import torch
import torch.nn as nn
from torch.nn.modules.module import _has_any_global_hook

from .. import _lib
from ..dualpipe_utils import FP8WeightCacheControl
from ..operators import fused_experts
from ..operators.clamped_swiglu import clamped_swiglu
from ..operators.deepgemm_quantize import fp8cast_grouped_weight, fp8cast_grouped_weight_cat, fp8cast_grouped_weights, weight_twin_enabled
from ..operators.grouped_linear import FP8GroupedLinear, FP8GroupedLinearFunc, GroupedLinearFunc
from ..operators.indexed_bias_add import indexed_bias_add
from ..operators.linear import FP8Linear
from ..operators.silu_mul import silu_mul, silu_mul_halves
from ..operators.token_scatter import (
    group_indices,
    group_rows_with_sizes,
    padded_index_gather,
    precompute_group_indices,
    scatter_for_grouped_gemm,
)
from . import training


def _weight(module: nn.Module, name: str = "weight") -> torch.Tensor:
    """``module.weight`` without the module's attribute search (a microsecond each, and a step of a small
    layer makes twenty of them).  A parametrised, pruned or sharded weight is no parameter of that name."""
    w = module._parameters.get(name)
    return w if w is not None else getattr(module, name)


def _cached(cache, version: int, now: int, twin: bool) -> bool:
    """Whether a module's cached quantised weight is of this version and has the twin that is asked for."""
    return cache is not None and version == now and (cache[2] is not None) == twin


def _whole_blocks(row_map, grouped_mm_offs):
    """Row map, group ends and group sizes of groups that are multiples of 64 rows, spread to multiples of 128.  A block is
    handed the former where nothing should be kept for a backward; if its forward finds otherwise (a pre-hook made the rows
    require a gradient, or changed their type), what runs then reads groups of whole 128-row tiles."""
    sizes = (torch.diff(grouped_mm_offs, prepend=grouped_mm_offs.new_zeros(1)) + 127) // 128 * 128
    ends = sizes.cumsum(0, dtype=torch.int32)
    rows = torch.arange(row_map.shape[0], device=row_map.device, dtype=torch.int32)
    moved = torch.cat([ends.new_zeros(1), ends - grouped_mm_offs])  # rows of padding before a group, and behind the last one
    at = rows + moved[torch.searchsorted(grouped_mm_offs, rows, right=True)]
    whole = row_map.new_full(((row_map.shape[0] + 64 * ends.shape[0] + 127) // 128 * 128,), -1)
    return whole.index_copy_(0, at.long(), row_map), ends, sizes


class Qwen3MoeExperts(nn.Module):
    def __init__(self, hidden_size: int, moe_intermediate_size: int, num_experts: int):
        super().__init__()
        self.gate_proj = training.GroupedLinear(num_experts, hidden_size, moe_intermediate_size)
        self.up_proj = training.GroupedLinear(num_experts, hidden_size, moe_intermediate_size)
        self.down_proj = training.GroupedLinear(num_experts, moe_intermediate_size, hidden_size)
        self._gu_cache = None  # gate and up quantised into one fused operand (FP8 path)
        self._gu_version = -1

    def _fused_gate_up_quant(self):
        """gate and up weights quantised into one fused ``[G, 2I, H]`` operand; cached like the
        layers' own quantised weights (one quantisation per ``FP8WeightCacheControl`` version)."""
        parts = [self.gate_proj.weight, self.up_proj.weight]
        if torch.compiler.is_compiling():
            return fp8cast_grouped_weight_cat(parts)
        ver = FP8WeightCacheControl.version
        if self._gu_cache is None or self._gu_version != ver or (self._gu_cache[2] is not None) != weight_twin_enabled():
            self._gu_cache = fp8cast_grouped_weight_cat(parts)
            self._gu_version = ver
        return self._gu_cache

    def _projections(self):
        m = self._modules
        return m["gate_proj"], m["up_proj"], m["down_proj"]

    def one_node(self, x) -> bool:
        """Whether the block runs as one autograd node on ``x``."""
        if not training.fp8 or x.dtype != torch.bfloat16:
            return False
        gate, up, down = self._projections()
        return (isinstance(gate, FP8GroupedLinear) and isinstance(up, FP8GroupedLinear) and isinstance(down, FP8GroupedLinear)
                and fused_experts.supported_split(x, _weight(gate), _weight(up), _weight(down)))

    def _quantized_weights(self):
        """The fused gate/up operand and the down operand, quantised by one launch when both are stale."""
        ver, twin = FP8WeightCacheControl.version, weight_twin_enabled()
        gate, up, down = self._projections()
        if torch.compiler.is_compiling():
            return self._fused_gate_up_quant(), down._get_quantized_weight()
        gu_ok = _cached(self._gu_cache, self._gu_version, ver, twin)
        down_ok = _cached(down._wq_cache, down._wq_version, ver, twin)
        if not (gu_ok or down_ok):
            self._gu_cache, down._wq_cache = fp8cast_grouped_weights([[_weight(gate), _weight(up)], [_weight(down)]])
            self._gu_version = down._wq_version = ver
        elif not (gu_ok and down_ok):
            return self._fused_gate_up_quant(), down._get_quantized_weight()
        return self._gu_cache, down._wq_cache

    def forward(self, x, grouped_mm_offs, ks=None, ks_tensor=None, row_map=None, fuse_activation: bool = True,
                expand_idx=None, few_rows: bool = False):
        """``row_map`` (extension, FP8 layers only): the scatter's int32 source-row map.  ``x`` is
        then the un-permuted ``[m, H]`` token tensor and the result comes back un-permuted; the
        permutation happens inside the first quantisation and the last GEMM's store.
        ``expand_idx`` (one-node path only): ``x`` holds deduplicated rows, see
        :func:`fused_experts.compose_row_maps`.  One-node path with ``row_map`` only: ``x`` may be an expanded
        ``[T, k, H]`` view of the tokens, and ``few_rows`` says that the groups are multiples of 64 rows (no
        backward may follow).  With ``fuse_activation`` (FP8 layers, intermediate size a multiple of 128) the block runs as one
        autograd node on a fused gate_up operand: the tokens are quantised once instead of once
        per projection, one GEMM serves both, and the SwiGLU and its gradient are computed inside
        the kernels that quantise them (same bits as the three-operator composition).  Asked here and not by the
        caller: a forward pre-hook may have changed ``x``."""
        if fuse_activation and x.shape[0] > 0 and self.one_node(x):
            gate, up, down = map(_weight, self._projections())
            if not fused_experts.wants_backward(x, gate, up, down):
                return fused_experts.forward_only(x, down, grouped_mm_offs, *self._quantized_weights(), row_map, expand_idx,
                                                  few_rows=few_rows)  # fmt: skip
            if few_rows:
                row_map, grouped_mm_offs, ks_tensor = _whole_blocks(row_map, grouped_mm_offs)
            return fused_experts.FP8SwiGLUSplitExpertsFunc.apply(
                x, gate, up, down, grouped_mm_offs, *self._quantized_weights(), row_map, expand_idx,
            )  # fmt: skip
        assert expand_idx is None, "expand_idx needs the one-node FP8 path"
        if few_rows:
            row_map, grouped_mm_offs, ks_tensor = _whole_blocks(row_map, grouped_mm_offs)
        gi = precompute_group_indices(grouped_mm_offs, x.shape[0])
        kwargs = dict(grouped_mm_offs=grouped_mm_offs, ks=ks, ks_tensor=ks_tensor, group_indices=gi)
        if row_map is not None:
            g = self.gate_proj(x, in_rows=row_map, **kwargs)
            u = self.up_proj(x, in_rows=row_map, **kwargs)
            return self.down_proj(silu_mul(g, u), out_rows=row_map, out_m=x.shape[0], **kwargs)
        g = self.gate_proj(x, **kwargs)
        u = self.up_proj(x, **kwargs)
        return self.down_proj(silu_mul(g, u), **kwargs)


class DeepSeekV2Experts(Qwen3MoeExperts):
    """Same composition as the Qwen3 experts (models/deepseek_v2.py:111-129)."""


class DeepSeekV2MLP(nn.Module):
    """Dense SwiGLU MLP (the shared experts run as one of these)."""

    def __init__(self, hidden_size: int, intermediate_size: int):
        super().__init__()
        self.gate_proj = training.Linear(hidden_size, intermediate_size, bias=False)
        self.up_proj = training.Linear(hidden_size, intermediate_size, bias=False)
        self.down_proj = training.Linear(intermediate_size, hidden_size, bias=False)
        self._q_cache = None  # the quantised weights of the one-node path, once per FP8WeightCacheControl version
        self._q_version = -1

    def _one_node(self, x: torch.Tensor):
        """The layer as one autograd node (gate and up as one fused operand, the SwiGLU and its gradient inside the
        quantisers), or None: not three plain FP8 linears, or shapes and types that the node does not take."""
        weights = []
        for m in self._modules.values():
            if (type(m) is not FP8Linear or m.bias is not None or m._forward_hooks or m._forward_pre_hooks or m._backward_hooks
                    or m._backward_pre_hooks or _has_any_global_hook()):
                return None
            weights.append(_weight(m))
        if len(weights) != 3 or x.dtype != torch.bfloat16 or not x.is_cuda or x.numel() == 0 or torch.compiler.is_compiling():
            return None
        ver = FP8WeightCacheControl.version
        x_2d = x if x.dim() == 2 else x.flatten(0, -2)
        out, quantised = _lib.host().mlp(x_2d, *weights, self._q_cache if self._q_version == ver else None, _lib.stream_ptr(x.device))
        if out is None:
            return None
        self._q_cache, self._q_version = quantised, ver
        return out if x.dim() == 2 else out.view(*x.shape[:-1], out.shape[-1])

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        out = self._one_node(x)
        return self.down_proj(silu_mul(self.gate_proj(x), self.up_proj(x))) if out is None else out


class Qwen35MoeExperts(nn.Module):
    def __init__(self, hidden_size: int, moe_intermediate_size: int, num_experts: int):
        super().__init__()
        self.num_experts = num_experts
        self.hidden_size = hidden_size
        self.moe_intermediate_size = moe_intermediate_size
        self.gate_up_proj = training.GroupedLinear(num_experts, hidden_size, 2 * moe_intermediate_size)
        self.down_proj = training.GroupedLinear(num_experts, moe_intermediate_size, hidden_size)

    def one_node(self, x) -> bool:
        """Whether the block runs as one autograd node on ``x``."""
        if not training.fp8 or x.dtype != torch.bfloat16:
            return False
        gate_up, down = self._modules["gate_up_proj"], self._modules["down_proj"]
        return (isinstance(gate_up, FP8GroupedLinear) and isinstance(down, FP8GroupedLinear)
                and fused_experts.supported(x, _weight(gate_up), _weight(down)))

    def _quantized_weights(self):
        """Both operands, quantised by one launch when both are stale."""
        ver, twin = FP8WeightCacheControl.version, weight_twin_enabled()
        gu, down = self._modules["gate_up_proj"], self._modules["down_proj"]
        if not torch.compiler.is_compiling():
            gu_ok = _cached(gu._wq_cache, gu._wq_version, ver, twin)
            down_ok = _cached(down._wq_cache, down._wq_version, ver, twin)
            if not (gu_ok or down_ok):
                gu._wq_cache, down._wq_cache = fp8cast_grouped_weights([[_weight(gu)], [_weight(down)]])
                gu._wq_version = down._wq_version = ver
                gu_ok = down_ok = True
            if gu_ok and down_ok:
                return gu._wq_cache, down._wq_cache
        return gu._get_quantized_weight(), down._get_quantized_weight()

    def forward(self, x, grouped_mm_offs, ks=None, ks_tensor=None, row_map=None, fuse_activation: bool = True,
                expand_idx=None, few_rows: bool = False):
        """``row_map`` / ``expand_idx``: see :meth:`Qwen3MoeExperts.forward`.  With ``fuse_activation`` (FP8 layers)
        the block runs as one autograd node whose SwiGLU output and SwiGLU gradient are computed
        inside the kernels that quantise them (same bits as the three-operator composition)."""
        if fuse_activation and x.shape[0] > 0 and self.one_node(x):
            gate_up, down = _weight(self._modules["gate_up_proj"]), _weight(self._modules["down_proj"])
            if not fused_experts.wants_backward(x, gate_up, down):
                return fused_experts.forward_only(x, down, grouped_mm_offs, *self._quantized_weights(), row_map, expand_idx,
                                                  few_rows=few_rows)  # fmt: skip
            if few_rows:
                row_map, grouped_mm_offs, ks_tensor = _whole_blocks(row_map, grouped_mm_offs)
            return fused_experts.FP8SwiGLUExpertsFunc.apply(
                x, gate_up, down, grouped_mm_offs, ks, ks_tensor,
                *self._quantized_weights(), row_map, expand_idx,
            )  # fmt: skip
        assert expand_idx is None, "expand_idx needs the one-node FP8 path"
        if few_rows:
            row_map, grouped_mm_offs, ks_tensor = _whole_blocks(row_map, grouped_mm_offs)
        gi = precompute_group_indices(grouped_mm_offs, x.shape[0])
        kwargs = dict(grouped_mm_offs=grouped_mm_offs, ks=ks, ks_tensor=ks_tensor, group_indices=gi)
        if row_map is not None:
            gate_up = self.gate_up_proj(x, in_rows=row_map, **kwargs)
            return self.down_proj(silu_mul_halves(gate_up), out_rows=row_map, out_m=x.shape[0], **kwargs)
        gate_up = self.gate_up_proj(x, **kwargs)
        # the halves are read in place (same arithmetic as silu_mul on contiguous copies)
        return self.down_proj(silu_mul_halves(gate_up), **kwargs)


class GptOssExperts(nn.Module):
    def __init__(self, hidden_size: int, intermediate_size: int, num_experts: int, swiglu_limit: float = 7.0):
        super().__init__()
        self.num_experts = num_experts
        self.swiglu_limit = float(swiglu_limit)
        self.gate_up_proj = nn.Parameter(torch.empty(num_experts, 2 * intermediate_size, hidden_size))
        self.gate_up_proj_bias = nn.Parameter(torch.zeros(num_experts, 2 * intermediate_size))
        self.down_proj = nn.Parameter(torch.empty(num_experts, hidden_size, intermediate_size))
        self.down_proj_bias = nn.Parameter(torch.zeros(num_experts, hidden_size))
        self._wq_cache: dict | None = None
        self._wq_version: int = -1
        # extension: the two indexed_bias_add steps happen in the stores of the GEMMs before them
        # (same bits) wherever the shapes and dtypes allow it
        self.fuse_bias = True
        # extension (needs fuse_bias): the whole block as one autograd node whose quantisation
        # kernels compute the clamped SwiGLU and its gradient instead of reading them from memory
        self.fuse_activation = True

    def _quantized_weight(self, name: str, weight: torch.Tensor):
        if torch.compiler.is_compiling():
            return fp8cast_grouped_weight(weight)
        ver = FP8WeightCacheControl.version
        cache = self._wq_cache
        if self._wq_version != ver or cache is None:
            cache = self._wq_cache = {}
            self._wq_version = ver
        if name not in cache or (cache[name][2] is not None) != weight_twin_enabled():
            cache[name] = fp8cast_grouped_weight(weight)
        return cache[name]

    def _quantized_weights(self):
        """Both operands, quantised by one launch when neither is cached."""
        stale = self._wq_version != FP8WeightCacheControl.version or not self._wq_cache
        if stale and not (torch.compiler.is_compiling() or weight_twin_enabled()):
            gate_up, down = fp8cast_grouped_weights([[self.gate_up_proj], [self.down_proj]])
            self._wq_cache = {"gate_up_proj": gate_up, "down_proj": down}
            self._wq_version = FP8WeightCacheControl.version
        return self._quantized_weight("gate_up_proj", self.gate_up_proj), self._quantized_weight("down_proj", self.down_proj)

    def _group_linear(self, x, weight, name, offs, ks, ks_tensor, group_indices_, in_rows=None, bias=None,
                      out_rows=None, out_m=None):
        if x.shape[0] == 0:
            return x @ weight[0].transpose(-2, -1)
        if training.fp8:
            return FP8GroupedLinearFunc.apply(
                x, weight, offs, ks, ks_tensor, self._quantized_weight(name, weight), group_indices_, in_rows,
                out_rows, out_m, bias,
            )
        assert in_rows is None, "row maps need the FP8 layers"
        return GroupedLinearFunc.apply(x, weight, offs)

    def bias_fusable(self, x) -> bool:
        """Whether the two ``indexed_bias_add`` steps happen in the stores of the GEMMs."""
        return (self.fuse_bias and training.fp8 and x.shape[0] > 0 and x.dtype == torch.bfloat16
                and _weight(self, "gate_up_proj_bias").dtype == x.dtype and _weight(self, "down_proj_bias").dtype == x.dtype
                and _weight(self, "gate_up_proj").shape[1] % 8 == 0 and _weight(self, "down_proj").shape[1] % 8 == 0)

    def one_node(self, x) -> bool:
        """Whether the block runs as one autograd node (fused biases and activation).  That node
        takes every row count from ``grouped_mm_offs`` on the device, so its ``row_map`` may be
        sized for more rows than the routing produced."""
        return self.bias_fusable(x) and self.fuse_activation and self.down_proj.shape[2] % 8 == 0

    def forward(self, x, grouped_mm_offs, ks=None, ks_tensor=None, row_map=None, scatter_output: bool = False,
                few_rows: bool = False):
        """``row_map`` (extension, FP8 only): the scatter's int32 source-row map; ``x`` is then the
        un-permuted token tensor and the first quantisation gathers its rows.  The result stays
        in the grouped layout unless ``scatter_output`` is set (with ``row_map`` and the fused
        biases): then the last GEMM stores every row, bias added, at its un-permuted place, and
        the backward sums the bias gradient over the grouped order through the same map.
        With ``self.fuse_bias`` (FP8 only) the two ``indexed_bias_add`` steps happen in the stores
        of the GEMMs before them (same bits)."""
        M = x.shape[0] if row_map is None else row_map.shape[0]
        fused = self.bias_fusable(x)
        assert not scatter_output or (fused and row_map is not None), "scatter_output needs row_map and the fused biases"
        if M % 128 == 0 and self.one_node(x):
            gate_up, gate_up_bias, down, down_bias = (_weight(self, n) for n in ("gate_up_proj", "gate_up_proj_bias", "down_proj", "down_proj_bias"))
            if not fused_experts.wants_backward(x, gate_up, gate_up_bias, down, down_bias):
                return fused_experts.forward_only(
                    x, down, grouped_mm_offs, *self._quantized_weights(), row_map, None, scatter_output,
                    (1.702, self.swiglu_limit), (gate_up_bias, down_bias), few_rows,
                )
            if few_rows:
                row_map, grouped_mm_offs, ks_tensor = _whole_blocks(row_map, grouped_mm_offs)
            return fused_experts.FP8ClampedSwiGLUExpertsFunc.apply(
                x, gate_up, gate_up_bias, down, down_bias, grouped_mm_offs,
                *self._quantized_weights(), 1.702, self.swiglu_limit, row_map, scatter_output,
            )
        if fused:
            gate_up = self._group_linear(x, self.gate_up_proj, "gate_up_proj", grouped_mm_offs, ks, ks_tensor, None, row_map,
                                         self.gate_up_proj_bias)
            activated = clamped_swiglu(gate_up, 1.702, self.swiglu_limit)
            return self._group_linear(activated, self.down_proj, "down_proj", grouped_mm_offs, ks, ks_tensor, None, None,
                                      self.down_proj_bias, row_map if scatter_output else None,
                                      x.shape[0] if scatter_output else None)
        group_ids = group_indices(grouped_mm_offs, M, torch.int64)
        gate_up = self._group_linear(x, self.gate_up_proj, "gate_up_proj", grouped_mm_offs, ks, ks_tensor, None, row_map)
        gate_up = indexed_bias_add(gate_up, self.gate_up_proj_bias, group_ids, grouped_mm_offs)
        activated = clamped_swiglu(gate_up, 1.702, self.swiglu_limit)
        out = self._group_linear(activated, self.down_proj, "down_proj", grouped_mm_offs, ks, ks_tensor, None)
        return indexed_bias_add(out, self.down_proj_bias, group_ids, grouped_mm_offs)


_ONE_NODE_BLOCKS = (Qwen3MoeExperts, Qwen35MoeExperts, GptOssExperts)


def _few_rows(experts: nn.Module, x, expert_idxs, experts_per_rank: int) -> bool:
    return (fused_experts.few_rows_per_expert(expert_idxs.shape[0], experts_per_rank)
            and not fused_experts.wants_backward(x, *experts.parameters()))


def forward_stage3(experts: nn.Module, gathered_tokens, expert_idxs, experts_per_rank: int, expand_idx=None,
                   fuse_expand: bool = True, fuse_permute: bool = True, host_sizes: bool = False):
    """Expert compute between the dispatch and combine all-to-alls.

    With ``fuse_permute`` (FP8 Qwen3 / DeepSeek / Qwen3.5 experts, no ``expand_idx``) the permuted
    copy of the tokens, its inverse gather and their two backward passes are never materialised:
    only the index half of the scatter runs, the first quantisation reads rows through the
    source map and the last GEMM of forward and of backward stores rows through it.  The result
    is bit-identical to the unfused composition.  Unless ``host_sizes`` is set, this path also
    drops the scatter's device-to-host copy of the group sizes (token_scatter.py:230-243 waits for
    the GPU there on every call): buffers are sized for the largest padded row count the routing
    could produce and every kernel reads the real count from ``grouped_mm_offs``.

    ``expand_idx`` (EP > 1) re-expands the deduplicated received rows to one row per routed
    (token, expert) pair.  With ``fuse_expand`` that gather is folded into the scatter's row copy
    (each unique row is read once per use and no expanded copy is materialised); without it the
    two steps run separately as in the reference.

    The block gets a keyword of an extension only in the calls that need it, so a subclass whose ``forward`` lacks
    ``expand_idx`` or ``few_rows`` runs wherever there is nothing to expand and a backward follows.

    ``gathered_tokens`` may also be an expanded ``[T, k, H]`` view of one row per token (stride 0 along k):
    the one-node blocks then read every token where it is, and its gradient comes back as ``[T, k, H]``.
    """
    if gathered_tokens.dim() == 3:
        T, k = gathered_tokens.shape[:2]
        one = (fuse_permute and training.fp8 and expand_idx is None and T > 0 and isinstance(experts, _ONE_NODE_BLOCKS)
               and experts.one_node(gathered_tokens[:, 0]) and gathered_tokens.stride(1) == 0 and T * k * k < 2**32)
        if not one:
            gathered_tokens = gathered_tokens.reshape(T * k, -1)
    if fuse_permute and training.fp8 and expert_idxs.shape[0] > 0 and isinstance(experts, (Qwen3MoeExperts, Qwen35MoeExperts)):
        fused_node = experts.one_node(gathered_tokens)
        # the composition of separate operators can still take the row map when its layers are FP8 ones
        down = experts._modules["down_proj"]
        mapped = fused_node or (isinstance(down, FP8GroupedLinear) and down.out_features % 8 == 0 and down.in_features % 8 == 0)
        if mapped and (expand_idx is None or (fused_node and fuse_expand)):
            few = fused_node and not host_sizes and _few_rows(experts, gathered_tokens, expert_idxs, experts_per_rank)
            _, grouped_mm_offs, ks, ks_tensor, src_of = group_rows_with_sizes(
                expert_idxs, experts_per_rank, fused_experts.FEW_ROWS if few else 128, device=gathered_tokens.device,
                host_sizes=host_sizes or not fused_node, need_reverse=False)
            # deduplicated rows: the first quantisation reads them through expand_idx composed with
            # the scatter's map, so neither the expanded nor the permuted copy exists
            return experts(gathered_tokens, grouped_mm_offs, ks=ks, ks_tensor=ks_tensor, row_map=src_of,
                           **({} if expand_idx is None else {"expand_idx": expand_idx}), **({"few_rows": True} if few else {}))
    if (fuse_permute and expand_idx is None and training.fp8 and expert_idxs.shape[0] > 0
            and isinstance(experts, GptOssExperts)):
        # the one-node block needs no host-side sizes (see the SwiGLU branch above)
        fused_node = experts.one_node(gathered_tokens)
        few = fused_node and not host_sizes and _few_rows(experts, gathered_tokens, expert_idxs, experts_per_rank)
        reverse_shuffle_idxs, grouped_mm_offs, ks, ks_tensor, src_of = group_rows_with_sizes(
            expert_idxs, experts_per_rank, fused_experts.FEW_ROWS if few else 128, device=gathered_tokens.device,
            host_sizes=host_sizes or not fused_node, need_reverse=not fused_node)
        if experts.bias_fusable(gathered_tokens):
            # both sides: rows gathered by the first quantisation, stored un-permuted (bias added)
            # by the last GEMM; the bias gradients are summed through the same map
            return experts(gathered_tokens, grouped_mm_offs, ks=ks, ks_tensor=ks_tensor, row_map=src_of, scatter_output=True,
                           **({"few_rows": True} if few else {}))
        # input side only: the unfused bias add wants the grouped layout
        outs = experts(gathered_tokens, grouped_mm_offs, ks=ks, ks_tensor=ks_tensor, row_map=src_of)
        return padded_index_gather(outs, reverse_shuffle_idxs)
    pre = None
    if expand_idx is not None:
        if fuse_expand:
            pre = expand_idx
        else:
            gathered_tokens = padded_index_gather(gathered_tokens, expand_idx)
    output_tokens, reverse_shuffle_idxs, grouped_mm_offs, ks, ks_tensor = scatter_for_grouped_gemm(
        gathered_tokens, expert_idxs, experts_per_rank, pre_index=pre
    )
    del gathered_tokens
    outs = experts(output_tokens, grouped_mm_offs, ks=ks, ks_tensor=ks_tensor)
    return padded_index_gather(outs, reverse_shuffle_idxs)
