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
