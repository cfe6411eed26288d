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


@pytest.mark.parametrize("width", [272, 512, 128])
def test_dense_linear_refuses_an_input_of_another_width(width):
    """With the weight quantised in the call and with a kept one; the backward's operands likewise."""
    from pith_train_amd._lib import PithTrainHipError
    from pith_train_amd.operators import linear as L

    m = L.FP8Linear(256, 128, bias=False, device="cuda", dtype=torch.bfloat16)
    for _ in range(2):
        with pytest.raises(PithTrainHipError, match="width"):
            m(_randn(32, width))
        m(_randn(32, 256)).sum().backward()
    _, _, w_t, w_ts = m._get_quantized_weight()
    heads = [_randn(32, 2, 32, grad=False), _randn(32, 2, 32, grad=False)]
    with pytest.raises(PithTrainHipError, match="transposed weight"):
        L.fp8_dgrad_wgrad_heads(*heads, w_t, w_ts, _randn(32, width, grad=False), width)
    x_t = torch.empty((256, 32), dtype=torch.float8_e4m3fn, device="cuda")
    with pytest.raises(PithTrainHipError, match="transposed weight"):
        L.fp8_dgrad_wgrad(_randn(32, 128, grad=False), w_t, w_ts, x_t, w_ts, 512)


def test_weights_and_indices_on_the_host_are_refused():
    from pith_train_amd._lib import PithTrainHipError
    from pith_train_amd.modules.experts import DeepSeekV2MLP, Qwen3MoeExperts, forward_stage3
    from pith_train_amd.operators.linear import FP8Linear
    from pith_train_amd.operators.token_scatter import scatter_for_grouped_gemm

    x = _randn(32, 128)
    for m in (DeepSeekV2MLP(128, 128).to(torch.bfloat16), FP8Linear(128, 128, bias=False, dtype=torch.bfloat16)):
        with pytest.raises(PithTrainHipError, match="GPU"):
            m(x)
    keys, pre = torch.randint(0, 4, (48,), device="cuda"), torch.randint(0, 32, (48,))
    with pytest.raises(PithTrainHipError, match="GPU"):
        scatter_for_grouped_gemm(x, keys, 4, pre_index=pre)
    experts = Qwen3MoeExperts(128, 128, 4).cuda().to(torch.bfloat16)
    with pytest.raises(PithTrainHipError, match="GPU"):
        forward_stage3(experts, x, keys, 4, expand_idx=pre)


@pytest.mark.parametrize("rows", [0, 5])
@pytest.mark.parametrize("expand", [False, True])
@pytest.mark.parametrize("family", ["Qwen3MoeExperts", "Qwen35MoeExperts", "GptOssExperts"])
def test_a_rank_without_rows_stays_in_the_graph(rows, expand, family):
    """The gradient of what it received is a zero tensor, so a linked all-to-all runs its backward there too."""
    from pith_train_amd.modules import experts as X

    m = getattr(X, family)(128, 128, 4).cuda().to(torch.bfloat16)
    received = _randn(rows, 128)
    none = torch.zeros((0,), dtype=torch.int64, device="cuda")
    out = X.forward_stage3(m, received * 1.0, none, 4, expand_idx=none if expand else None)
    assert out.shape == (0, 128) and out.requires_grad
    (grad,) = torch.autograd.grad(out, received, torch.zeros_like(out))
    assert grad.shape == received.shape and not grad.any()


@pytest.mark.parametrize("train", [True, False])
def test_gpt_oss_block_refuses_biases_and_weights_of_other_shapes(train):
    from pith_train_amd._lib import PithTrainHipError
    from pith_train_amd.modules.experts import GptOssExperts, Qwen3MoeExperts, forward_stage3

    keys = torch.randint(0, 4, (48,), device="cuda")

    def refused(error, m, width=128):
        with torch.set_grad_enabled(train), pytest.raises(error):
            forward_stage3(m, _randn(48, width, grad=train), keys, 4)

    for name, shape in (("gate_up_proj_bias", (4, 128)), ("gate_up_proj_bias", (3, 256)), ("down_proj_bias", (4, 64)), ("down_proj_bias", (1, 128))):
        m = GptOssExperts(128, 128, 4).cuda().to(torch.bfloat16)
        setattr(m, name, torch.nn.Parameter(torch.zeros(shape, device="cuda", dtype=torch.bfloat16)))
        refused(AssertionError, m)
    refused(PithTrainHipError, GptOssExperts(128, 128, 4).cuda().to(torch.bfloat16), 256)
    refused(PithTrainHipError, Qwen3MoeExperts(128, 128, 4).cuda().to(torch.bfloat16), 256)
    refused(PithTrainHipError, Qwen3MoeExperts(128, 128, 3).cuda().to(torch.bfloat16))


def _hidden_activations(kind):
    """(module call, input, bytes of the activations that the backward needs besides weights)"""
    from pith_train_amd.modules import experts as X
    from pith_train_amd.operators.linear import FP8Linear
    from pith_train_amd.operators.token_scatter import scatter_for_grouped_gemm

    T, H, half, E = 300, 256, 384, 4
    if kind == "mlp":
        m = X.DeepSeekV2MLP(H, half)
        return m, m, T * (H + 2 * 2 * half + half)
    if kind == "linear":
        m = FP8Linear(H, half, bias=False)
        return m, m, T * H
    keys = torch.randint(0, E, (T,), device="cuda")
    if kind == "grouped":
        m = X.Qwen3MoeExperts(H, half, E)

        def call(x):
            rows, reverse, offs, ks, ks_t = scatter_for_grouped_gemm(x, keys, E)
            return m.gate_proj(rows, grouped_mm_offs=offs, ks=ks, ks_tensor=ks_t)

        return m, call, T * H
    m = getattr(X, kind)(H, half, E)
    return m, lambda x: X.forward_stage3(m, x, keys, E), T * (H + 2 * 2 * half + half)


@pytest.mark.parametrize("kind", ["Qwen3MoeExperts", "Qwen35MoeExperts", "GptOssExperts", "grouped", "mlp", "linear"])
def test_hooks_on_saved_tensors_see_the_activations(kind):
    """save_on_cpu and checkpointing without re-entry can let go of what a layer keeps: same gradients, nothing of it
    left on the GPU in between."""
    from torch.utils.checkpoint import checkpoint

    m, call, nbytes = _hidden_activations(kind)
    m.cuda().to(torch.bfloat16)
    with torch.no_grad():
        for p in m.parameters():
            p.normal_(0.0, 0.05)
    x = _randn(300, 256)

    def step(forward):
        m.zero_grad(set_to_none=True)
        out = forward(x)
        dy = torch.linspace(-1, 1, out.numel(), device="cuda").view(out.shape).to(out.dtype)
        grads = torch.autograd.grad(out, [x, *m.parameters()], dy, allow_unused=True)
        return [out.detach(), *[p.grad if g is None else g for p, g in zip([None, *m.parameters()], grads) if g is not None or p.grad is not None]]

    def offloaded(x):
        seen = []

        def pack(t):
            seen.append(t.numel() * t.element_size())
            return t.cpu()

        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
            out = call(x)
        assert sum(seen) >= nbytes
        return out

    want = step(call)
    for forward in (offloaded, lambda x: checkpoint(call, x, use_reentrant=False)):
        got = step(forward)
        assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.reshape(-1)[:1]):
        out = call(x)
    with pytest.raises(RuntimeError):
        out.sum().backward()


@pytest.mark.parametrize("kind", ["linear", "mlp", "grouped"])
@pytest.mark.parametrize("fresh", [True, False])
def test_rows_that_share_memory(kind, fresh):
    """An input and a gradient of one row for all: a broadcast, and a sum over the rows."""
    from pith_train_amd.dualpipe_utils import FP8WeightCacheControl
    from pith_train_amd.modules import experts as X
    from pith_train_amd.operators.linear import FP8Linear

    offs = torch.tensor([128, 256], dtype=torch.int32, device="cuda")
    m = {"linear": lambda: FP8Linear(256, 128, bias=False), "mlp": lambda: X.DeepSeekV2MLP(256, 256),
         "grouped": lambda: X.FP8GroupedLinear(2, 256, 128)}[kind]().cuda().to(torch.bfloat16)
    with torch.no_grad():
        for p in m.parameters():
            p.normal_(0.0, 0.05)
    call = (lambda x: m(x, grouped_mm_offs=offs)) if kind == "grouped" else m

    def step(shared):
        if fresh:
            FP8WeightCacheControl.step()
        m.zero_grad(set_to_none=True)
        x = _randn(1, 256).detach().fill_(0.5).requires_grad_(True)
        rows = x.expand(256, 256)
        out = call(rows if shared else rows.contiguous())
        dy = torch.linspace(-1, 1, out.shape[1], device="cuda").bfloat16().expand(out.shape)
        out.backward(dy if shared else dy.contiguous())
        return [out.detach(), x.grad, *(p.grad for p in m.parameters())]

    assert all(torch.equal(a, b) for a, b in zip(step(True), step(False)))


class _Doubled(torch.nn.Module):
    def forward(self, w):
        return 2.0 * w


@pytest.mark.parametrize("family,names", [("Qwen3MoeMoE", ["gate.weight"]), ("DeepSeekV2MoE", ["gate.weight", "shared_experts.up_proj.weight"]),
                                          ("GptOssMoE", ["router.weight", "experts.down_proj_bias"])])
def test_block_with_parametrised_weights(family, names):
    """Twice the stored weight equals a block that stores twice the weight; the gradient reaches the stored one."""
    from torch.nn.utils import parametrize

    from pith_train_amd.dualpipe_utils import FP8WeightCacheControl
    from pith_train_amd.modules import moe

    torch.manual_seed(1)
    block = getattr(moe, family)(128, 128, 8, 2).cuda().to(torch.bfloat16)
    with torch.no_grad():
        for p in block.parameters():
            p.normal_(0.0, 0.05)
    x = _randn(64, 128, grad=False)
    for name in names:
        module, attr = block.get_submodule(name.rpartition(".")[0]), name.rpartition(".")[2]
        w = getattr(module, attr)
        with torch.no_grad():
            w.mul_(2.0)
        FP8WeightCacheControl.step()
        want = block.reference_forward(x)
        with torch.no_grad():
            w.mul_(0.5)
        parametrize.register_parametrization(module, attr, _Doubled())
        FP8WeightCacheControl.step()
        got = block.reference_forward(x)
        torch.testing.assert_close(got, want, rtol=2.0**-7, atol=2.0**-7 * want.float().abs().max().item())
        (grad,) = torch.autograd.grad(got.float().square().sum(), getattr(module.parametrizations, attr).original, allow_unused=False)
        assert grad.abs().sum() > 0
        parametrize.remove_parametrizations(module, attr, leave_parametrized=False)


def test_gate_and_branches_are_differentiable_twice_and_forward():
    """As the torch expressions they stand for: the gate's product, and the input handed to several consumers."""
    import torch.nn.functional as F
    from torch.autograd import forward_ad

    from pith_train_amd.modules.gates import DeepSeekV2MoEGate, Qwen3MoeGate
    from pith_train_amd.operators.moe_combine import token_branches

    for make, fp32 in ((Qwen3MoeGate, False), (DeepSeekV2MoEGate, True)):
        gate = make(8, 64, 2).cuda().to(torch.bfloat16)
        torch.nn.init.normal_(gate.weight)
        x, up = _randn(40, 64), torch.randn((40, 8), device="cuda")
        results = []
        for logits in (gate._logits(x, fp32), F.linear(x.float(), gate.weight.float()) if fp32 else F.linear(x, gate.weight)):
            gx, gw = torch.autograd.grad(logits, [x, gate.weight], (up.to(logits.dtype) * logits), create_graph=True)
            results.append([logits, gx, gw, *torch.autograd.grad(gx.float().square().sum() + gw.float().square().sum(), [x, gate.weight])])
        for got, want in zip(*results):
            torch.testing.assert_close(got, want, rtol=0.02, atol=0.02 * want.float().abs().max().item())
        with forward_ad.dual_level():
            dual = forward_ad.make_dual(x.detach(), torch.ones_like(x))
            tangent = forward_ad.unpack_dual(gate._logits(dual, fp32)).tangent
            assert tangent is not None and torch.equal(tangent[0], tangent[1])
            assert all(forward_ad.unpack_dual(b).tangent is not None for b in token_branches(dual.requires_grad_(True), 2, 1))


@pytest.mark.parametrize("kind", ["Qwen3MoeExperts", "grouped", "mlp", "linear"])
def test_what_a_kernel_cannot_differentiate_is_refused(kind):
    """Not dropped: a second derivative, and a forward-mode one."""
    from torch.autograd import forward_ad

    m, call, _ = _hidden_activations(kind)
    m.cuda().to(torch.bfloat16)
    with torch.no_grad():
        for p in m.parameters():
            p.normal_(0.0, 0.05)
    x = _randn(300, 256)
    out = call(x)
    (grad,) = torch.autograd.grad(out, x, torch.ones_like(out), create_graph=True)
    assert grad.requires_grad
    with pytest.raises(RuntimeError, match="cannot be differentiated"):
        grad.sum().backward()
    with forward_ad.dual_level(), pytest.raises(RuntimeError, match="forward-mode|forward mode|forward AD"):
        call(forward_ad.make_dual(x.detach(), torch.ones_like(x)).requires_grad_(True))
    with torch.no_grad(), forward_ad.dual_level(), pytest.raises(RuntimeError, match="forward-mode|forward mode|forward AD"):
        call(forward_ad.make_dual(x.detach(), torch.ones_like(x)))


def test_errors_of_a_backward_keep_their_types(monkeypatch):
    from pith_train_amd import _lib
    from pith_train_amd.dualpipe_utils import WeightGradStore
    from pith_train_amd.modules.experts import Qwen3MoeExperts, forward_stage3
    from pith_train_amd.operators.silu_mul import silu_mul
    from pith_train_amd.operators.token_scatter import padded_index_gather

    out = padded_index_gather(_randn(6, 16, dtype=torch.float64), torch.randint(0, 6, (10,), device="cuda"))
    with pytest.raises(TypeError, match="dtype"):  # rows of any type are copied, but not summed
        out.sum().backward()
    out = silu_mul(_randn(4, 16), _randn(4, 16))
    with pytest.raises(AssertionError, match="contiguous"):
        out.backward(torch.ones((16, 4), device="cuda", dtype=torch.bfloat16).t())
    keys = torch.randint(0, 4, (48,), device="cuda")
    monkeypatch.setenv("PITHTRAIN_FP8_WEIGHT_TWIN", "1")
    out = forward_stage3(Qwen3MoeExperts(128, 128, 4).cuda().to(torch.bfloat16), _randn(48, 128), keys, 4)
    _lib.call("pt_gemm_select_kernel", b"t")  # a kernel that has no scattered store, which the host says
    try:
        with pytest.raises(_lib.PithTrainHipError, match="scattered"):
            out.sum().backward(retain_graph=True)
    finally:
        _lib.call("pt_gemm_select_kernel", None)

    def full(_):
        raise KeyError("queue")

    monkeypatch.setattr(WeightGradStore, "enabled", True)
    monkeypatch.setattr(WeightGradStore, "put", full)
    with pytest.raises(KeyError, match="queue"):
        out.sum().backward()


@pytest.mark.parametrize("hidden,inter", [(1024, 256), (512, 1024)])
def test_peak_memory_of_an_expert_block_backward(hidden, inter):
    """The row-scaled gradients and the activation's gradient are not held at once, nor with the last weight gradients:
    the largest phase is the activation's backward (its own buffers, both transposed gradients, the first weight
    gradient) or the one after it (the input gradient and the other weight gradients beside the transposed ones)."""
    from pith_train_amd.modules.experts import Qwen35MoeExperts, forward_stage3

    E, T = 4, 16384
    m = Qwen35MoeExperts(hidden, inter, E).cuda().to(torch.bfloat16)
    x, keys = _randn(T, hidden), torch.randint(0, E, (T,), device="cuda")
    out = forward_stage3(m, x, keys, E)
    dy = torch.ones_like(out)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    grad = torch.autograd.grad(out, x, dy)
    torch.cuda.synchronize()
    peak = torch.cuda.max_memory_allocated() - before
    rows = -(-(T + 127 * E) // 128) * 128 + 128
    transposed, down = rows * (hidden + 2 * inter), 2 * E * hidden * inter
    first = rows * (max(hidden, 2 * inter) + 2 * inter) + down
    second = rows * max(hidden, 2 * inter) + 2 * T * hidden + down
    third = 2 * T * hidden + 3 * down
    assert peak <= 1.05 * (transposed + max(first, second, third)) + (4 << 20), (peak, transposed, first, second, third)
    assert grad[0].shape == x.shape


def test_indices_of_other_types_and_lengths_are_refused():
    """They go to kernels by address."""
    from pith_train_amd.operators.ep_dispatch import adjust_expand_idx
    from pith_train_amd.operators.token_scatter import padded_index_gather, scatter_for_grouped_gemm

    x = _randn(6, 16)
    index = torch.randint(0, 6, (20,), device="cuda")
    with pytest.raises(TypeError, match="int64"):
        padded_index_gather(x, index.int())
    with pytest.raises(TypeError, match="int64"):
        scatter_for_grouped_gemm(x, index % 4, 4, pre_index=index.int())
    for keys, pre in ((index % 4, None), (index % 4, index[:10])):
        with pytest.raises(AssertionError, match="rows"):
            scatter_for_grouped_gemm(x, keys, 4, pre_index=pre)
    counts = torch.tensor([2, 4], device="cuda")
    with pytest.raises(TypeError, match="int64"):
        adjust_expand_idx(index[:6].int(), counts, counts)
    # a strided index is read as what it is
    rows, reverse, *_ = scatter_for_grouped_gemm(x, index[::2] % 4, 4, pre_index=index[::2])
    want = scatter_for_grouped_gemm(x, index[::2].contiguous() % 4, 4, pre_index=index[::2].contiguous())
    assert torch.equal(rows, want[0]) and torch.equal(reverse, want[1])


def test_kept_weights_and_repeated_rows_of_other_shapes_are_refused():
    """A weight replaced under a cache that still counts as fresh; [T, k, H] rows that are not one row k times."""
    from pith_train_amd._lib import PithTrainHipError
    from pith_train_amd.modules.experts import DeepSeekV2MLP, Qwen3MoeExperts, forward_stage3
    from pith_train_amd.operators.linear import FP8Linear
    from pith_train_amd.operators.token_scatter import group_rows_with_sizes

    mlp = DeepSeekV2MLP(128, 256).cuda().to(torch.bfloat16)
    mlp(_randn(32, 128))
    for m in (mlp.gate_proj, mlp.up_proj, mlp.down_proj):
        m.weight = torch.nn.Parameter(torch.zeros((128, 128), device="cuda", dtype=torch.bfloat16))
    with pytest.raises(PithTrainHipError, match="quantised"):
        mlp(_randn(32, 128))
    lin = FP8Linear(128, 64, bias=False, device="cuda", dtype=torch.bfloat16)
    lin(_randn(32, 128))
    q = list(lin._wq_cache)
    q[1] = q[1][:, :0]
    lin._wq_cache = tuple(q)
    with pytest.raises(PithTrainHipError, match="scales"):
        lin(_randn(32, 128))
    experts, x = Qwen3MoeExperts(128, 128, 4).cuda().to(torch.bfloat16), _randn(24, 2, 128)
    keys = torch.randint(0, 4, (48,), device="cuda")
    _, offs, _, ks, src = group_rows_with_sizes(keys, 4, host_sizes=False)
    for grad in (True, False):
        with torch.set_grad_enabled(grad), pytest.raises(AssertionError, match="expanded"):
            experts(x, offs, row_map=src)
    assert forward_stage3(experts, x, keys, 4).shape == (48, 128)  # there such rows are copied


def test_weights_replaced_under_a_kept_quantisation_are_refused():
    """Their gradients would be written past a smaller tensor."""
    from pith_train_amd._lib import PithTrainHipError
    from pith_train_amd.modules.experts import Qwen3MoeExperts, Qwen35MoeExperts, forward_stage3

    keys = torch.randint(0, 4, (48,), device="cuda")
    for make, name, shape in ((Qwen3MoeExperts, "gate_proj", (4, 128, 64)), (Qwen3MoeExperts, "up_proj", (4, 128, 64)), (Qwen35MoeExperts, "gate_up_proj", (2, 256, 128))):
        m = make(128, 128, 4).cuda().to(torch.bfloat16)
        forward_stage3(m, _randn(48, 128), keys, 4)
        for p in ("gate_proj", "up_proj") if make is Qwen3MoeExperts and name == "gate_proj" else (name,):
            getattr(m, p).weight = torch.nn.Parameter(torch.zeros(shape, device="cuda", dtype=torch.bfloat16))
        with pytest.raises((PithTrainHipError, AssertionError, RuntimeError)):
            forward_stage3(m, _randn(48, 128), keys, 4)
    m = Qwen3MoeExperts(128, 128, 2).cuda().to(torch.bfloat16)
    kw = dict(grouped_mm_offs=torch.tensor([128, 256], dtype=torch.int32, device="cuda"))
    m.gate_proj(_randn(256, 128), **kw)
    m.gate_proj.weight = torch.nn.Parameter(torch.zeros((2, 64, 128), device="cuda", dtype=torch.bfloat16))
    with pytest.raises(PithTrainHipError, match="another size"):
        m.gate_proj(_randn(256, 128), **kw)
