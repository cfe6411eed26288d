"""What the C++ autograd nodes (``csrc/host.cpp``) owe a caller besides their numbers: the errors, hooks and links of
an ordinary autograd node.  Everything here runs without a GPU: no launch is reached."""

import pytest
import torch
import torch.nn.functional as F


def _host():
    from pith_train_amd import _lib

    return _lib.host()


def test_input_of_a_block_written_before_its_backward_is_found_out():
    """hidden += block(hidden): the gate saved its branch of ``hidden``, whose values are gone."""
    x = torch.randn((6, 16), requires_grad=True)
    w = torch.randn((4, 16), requires_grad=True)
    hidden = x * 1.0
    _, for_gate, _ = _host().branches(hidden, 3, 2, 0)
    logits = F.linear(for_gate, w)
    hidden += 100.0
    assert for_gate._version == hidden._version
    with pytest.raises(RuntimeError, match="inplace"):
        torch.autograd.grad(logits.sum(), w)


def test_a_branch_of_a_block_cannot_be_written():
    for i in range(3):
        branch = _host().branches(torch.randn((6, 16), requires_grad=True) * 1.0, 3, 2, 0)[i]
        with pytest.raises(RuntimeError, match="inplace"):
            branch += 1.0


def test_branches_are_differentiable_twice():
    x = torch.randn((5, 8), dtype=torch.float64, requires_grad=True)
    assert torch.autograd.gradcheck(lambda t: _host().branches(t, 3, 2, 0), x)
    assert torch.autograd.gradgradcheck(lambda t: [b * b for b in _host().branches(t, 3, 2, 0)], x)


class _Doubled(torch.nn.Module):
    def forward(self, w):
        return 2.0 * w


def test_gates_and_experts_with_a_parametrised_weight():
    """The parameter is then no entry of that name, and the attribute computes the weight."""
    from torch.nn.utils import parametrize

    from pith_train_amd.modules.experts import GptOssExperts
    from pith_train_amd.modules.gates import Qwen3MoeGate

    gate = Qwen3MoeGate(4, 16, 2)
    torch.nn.init.normal_(gate.weight)
    x, w = torch.randn((6, 16)), gate.weight.detach().clone()
    parametrize.register_parametrization(gate, "weight", _Doubled())
    torch.testing.assert_close(gate._logits(x), F.linear(x, 2.0 * w))
    experts = GptOssExperts(16, 16, 2).to(torch.bfloat16)
    fusable = experts.bias_fusable(x.bfloat16())
    for name in ("gate_up_proj", "down_proj_bias"):
        parametrize.register_parametrization(experts, name, _Doubled())
    assert experts.bias_fusable(x.bfloat16()) == fusable


def test_import_leaves_the_process_as_it_is():
    """A library that is imported changes no setting of autograd's, nor of anything else the whole program uses."""
    import os
    import subprocess
    import sys

    code = """
import torch
def state():
    return (torch._C._is_multithreading_enabled(), torch.is_grad_enabled(), torch.get_num_threads(), torch.get_default_dtype(),
            torch.backends.cuda.matmul.allow_tf32, torch.are_deterministic_algorithms_enabled(), torch.is_anomaly_enabled())
before = state()
import pith_train_amd
from pith_train_amd import _lib
from pith_train_amd.modules import moe
_lib.host()
assert state() == before, (before, state())
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    subprocess.run([sys.executable, "-c", code], check=True, cwd=root)


def _grouped(expert_idxs, num_groups, alignment=128, **_):
    """The scatter's index half in torch: (reverse, ends, sizes on the host and the device, source row of every grouped row)."""
    sizes = torch.bincount(expert_idxs, minlength=num_groups)
    ks = (sizes + alignment - 1) // alignment * alignment
    ends = ks.cumsum(0).int()
    src_of = torch.full((-(-int(ks.sum()) // 128) * 128,), -1, dtype=torch.int32)
    for e in range(num_groups):
        rows = (expert_idxs == e).nonzero().flatten().int()
        src_of[int(ends[e] - ks[e]) :][: len(rows)] = rows
    return None, ends, ks.tolist(), ks.int(), src_of


class _InTorch:
    """A user's projection: an ``FP8GroupedLinear`` by type, with a forward of its own that takes any floating type."""

    def forward(self, input, grouped_mm_offs, ks=None, ks_tensor=None, group_indices=None, in_rows=None, out_rows=None, out_m=None):
        rows = input if in_rows is None else input[in_rows.long().clamp(min=0)]
        group = torch.searchsorted(grouped_mm_offs, torch.arange(len(rows), dtype=torch.int32), right=True).clamp(max=self.num_groups - 1)
        y = torch.einsum("mk,mnk->mn", rows, self.weight[group].to(rows.dtype))
        if out_rows is None:
            return y
        kept = (out_rows >= 0) & (torch.arange(len(out_rows)) < grouped_mm_offs[-1])
        return y.new_zeros((out_m, y.shape[1])).index_copy(0, out_rows[kept].long(), y[kept])


@pytest.mark.parametrize("family", ["Qwen3MoeExperts", "Qwen35MoeExperts"])
def test_a_hook_that_changes_the_rows_type_gets_the_composition(family, monkeypatch):
    """A block decides by the rows that its forward receives.  Behind this pre-hook they are no bf16 rows any more, so the
    separate projections, which may take them, run in the place of the one node."""
    from pith_train_amd.modules import experts as X
    from pith_train_amd.operators.grouped_linear import FP8GroupedLinear

    monkeypatch.setattr(X, "group_rows_with_sizes", _grouped)
    monkeypatch.setattr(X, "silu_mul", lambda g, u: F.silu(g) * u)
    monkeypatch.setattr(X, "silu_mul_halves", lambda y: F.silu(y[:, : y.shape[1] // 2]) * y[:, y.shape[1] // 2 :])
    torch.manual_seed(0)
    m = getattr(X, family)(16, 128, 3).to(torch.bfloat16)
    projection = type("Projection", (_InTorch, FP8GroupedLinear), {})
    for child in m.children():
        child.__class__ = projection
        torch.nn.init.normal_(child.weight, std=0.1)
    m.register_forward_pre_hook(lambda module, args: (args[0].float(), *args[1:]))
    x, expert_idxs = torch.randn((300, 16)).bfloat16(), torch.randint(0, 3, (300,))
    assert m.one_node(x)
    out = X.forward_stage3(m, x, expert_idxs, 3)
    w = [p.float() for p in m.parameters()]
    gate, up = (w[0], w[1]) if len(w) == 3 else (w[0][:, :128], w[0][:, 128:])
    want = torch.stack([w[-1][e] @ (F.silu(gate[e] @ t) * (up[e] @ t)) for e, t in zip(expert_idxs, x.float())])
    torch.testing.assert_close(out, want)


@pytest.mark.parametrize("family", ["Qwen3MoeExperts", "Qwen35MoeExperts", "GptOssExperts"])
def test_stage3_passes_an_extension_s_keyword_only_where_it_is_needed(family, monkeypatch):
    """A subclass whose forward has fewer of them trains; evaluation with few rows and deduplicated rows name theirs."""
    from pith_train_amd.modules import experts as X

    seen = []

    def forward(self, x, grouped_mm_offs, ks=None, ks_tensor=None, row_map=None, **extra):
        seen.append(extra)
        return x

    m = type("Narrow", (getattr(X, family),), {"forward": forward})(16, 128, 3).to(torch.bfloat16)
    monkeypatch.setattr(X, "group_rows_with_sizes", _grouped)
    x, expert_idxs = torch.randn((30, 16)).bfloat16(), torch.randint(0, 3, (30,))
    always = {"scatter_output": True} if family == "GptOssExperts" else {}
    X.forward_stage3(m, x, expert_idxs, 3)
    with torch.no_grad():
        X.forward_stage3(m, x, expert_idxs, 3)
    assert seen == [always, {**always, "few_rows": True}]
    if not always:
        X.forward_stage3(m, x, expert_idxs, 3, expand_idx=expert_idxs)
        assert seen[2].keys() == {"expand_idx"}


def test_groups_of_64_rows_spread_to_whole_blocks():
    """Every group starts at the end of the last one, padded to 128 rows, and has the same rows in the same order."""
    from pith_train_amd.modules.experts import _whole_blocks

    expert_idxs = torch.cat([torch.full((n,), e) for e, n in enumerate((1, 0, 64, 65, 128, 0, 200, 3))])
    expert_idxs = expert_idxs[torch.randperm(len(expert_idxs), generator=torch.Generator().manual_seed(0))]
    _, ends, _, _, few = _grouped(expert_idxs, 8, 64)
    _, want_ends, _, want_sizes, want = _grouped(expert_idxs, 8)
    got, got_ends, got_sizes = _whole_blocks(torch.cat([few, few.new_full((256,), -1)]), ends)  # longer than the grouped rows
    assert got_ends.dtype == torch.int32 and torch.equal(got_ends, want_ends) and torch.equal(got_sizes, want_sizes) and len(got) % 128 == 0
    assert torch.equal(got[: len(want)], want) and (got[len(want) :] == -1).all()
