"""The C++ autograd nodes (``csrc/host.cpp``) as autograd nodes: saved tensors that were written since, hooks on
saved tensors, links of ranks without rows, refused calls."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _randn(*shape, dtype=torch.bfloat16, grad=True):
    return torch.randn(shape, device="cuda").to(dtype).requires_grad_(grad)


def _combine():
    from pith_train_amd.operators.moe_combine import moe_combine

    outs, w = _randn(12, 16) * 1, _randn(4, 3, dtype=torch.float32) * 1
    return moe_combine(outs, w), [outs, w]


def _combine_ep():
    from pith_train_amd.operators.moe_combine import moe_combine_ep

    outs, w, slots = _randn(12, 16) * 1, _randn(4, 3, dtype=torch.float32) * 1, torch.randperm(12, device="cuda")
    return moe_combine_ep(outs, slots, w, _randn(4, 16)), [outs, w]


def _router():
    from pith_train_amd.operators.router_topk import softmax_topk

    logits = _randn(8, 16, dtype=torch.float32) * 1
    idx, weight = softmax_topk(logits, 2)
    return weight, [logits, idx]


def _gather():
    from pith_train_amd.operators.token_scatter import padded_index_gather

    index = torch.randint(0, 6, (10,), device="cuda")
    return padded_index_gather(_randn(6, 16), index), [index]


def _scatter():
    from pith_train_amd.operators.token_scatter import scatter_for_grouped_gemm

    keys, pre = torch.randint(0, 4, (10,), device="cuda"), torch.randint(0, 6, (10,), device="cuda")
    rows, reverse, *_ = scatter_for_grouped_gemm(_randn(6, 16), keys, 4, pre_index=pre)
    return rows, [reverse, pre]


@pytest.mark.parametrize("make", [_combine, _combine_ep, _router, _gather, _scatter])
def test_saved_tensors_written_before_the_backward_are_found_out(make):
    for i in range(len(make()[1])):
        out, saved = make()
        with torch.no_grad():
            saved[i].mul_(1)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            out.sum().backward()
    out, _ = make()
    out.sum().backward()


def test_results_of_the_scatter_are_written_independently():
    from pith_train_amd.operators.token_scatter import scatter_for_grouped_gemm

    x = _randn(10, 16)
    rows, reverse, offs, ks, ks_tensor = scatter_for_grouped_gemm(x, torch.randint(0, 4, (10,), device="cuda"), 4)
    version = offs._version
    ks_tensor.add_(1)
    assert offs._version == version and int(offs[-1]) == sum(ks)
    rows.sum().backward()
