"""GPU tests of a MoE block's evaluation forward (nothing kept, groups of 64 rows), of the rows its experts
read without copies, and of the sum of its branches' gradients."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _block(family, H, I, E, k, seed):
    from pith_train_amd.modules import moe as M

    make = {"qwen3": lambda: M.Qwen3MoeMoE(H, I, E, k), "deepseek_v2": lambda: M.DeepSeekV2MoE(H, I, E, k, n_shared_experts=1),
            "gpt_oss": lambda: M.GptOssMoE(H, I, E, k), "qwen35": lambda: M.Qwen35MoeSparseMoeBlock(H, I, E, k, I)}[family]
    blk = make().cuda().to(torch.bfloat16)
    g = torch.Generator(device="cuda").manual_seed(seed)
    with torch.no_grad():
        for p in blk.parameters():
            p.normal_(0.0, 0.05, generator=g)
    return blk, g


@pytest.mark.parametrize("family", ["qwen3", "deepseek_v2", "gpt_oss", "qwen35"])
@pytest.mark.parametrize("T,E,k", [(1, 8, 2), (65, 8, 3), (192, 4, 1), (193, 16, 4), (700, 8, 2)])
def test_evaluation_forward_has_the_bits_of_the_training_forward(family, T, E, k):
    """Below and above the row count up to which evaluation pads its groups to 64 rows, with one choice per
    token (nothing repeated) and top-k counts that are no power of two."""
    from pith_train_amd.operators.fused_experts import few_rows_per_expert

    blk, g = _block(family, 256, 128 if family != "gpt_oss" else 144, E, k, T)
    assert few_rows_per_expert(T * k, E) == (T < 700 and T * k <= 48 * E)
    x = torch.randn((T, 256), generator=g, device="cuda").bfloat16()
    want = blk.reference_forward(x)
    assert want.requires_grad
    with torch.no_grad():
        got = blk.reference_forward(x)
    assert torch.equal(got, want.detach())


@pytest.mark.parametrize("rows,repeat,H", [(1, 2, 128), (100, 3, 264), (257, 6, 256), (64, 8, 2048)])
@pytest.mark.parametrize("twin", [True, False])
def test_rows_read_through_a_repeat_equal_the_repeated_rows(rows, repeat, H, twin):
    from pith_train_amd import _lib
    from pith_train_amd.operators.deepgemm_quantize import fp8cast_rowwise_colwise_t_rows

    M = -(-rows * repeat // 128) * 128 + 128
    g = torch.Generator().manual_seed(rows)
    x = torch.randn((rows, H), generator=g).bfloat16().cuda()
    index = torch.full((M,), -1, dtype=torch.int32)
    index[torch.randperm(M, generator=g)[: rows * repeat]] = torch.arange(rows * repeat, dtype=torch.int32)
    index = index.cuda()
    want = fp8cast_rowwise_colwise_t_rows(x.repeat_interleave(repeat, 0), index)
    got = [torch.zeros_like(t.view(torch.uint8) if t.dtype == torch.float8_e4m3fn else t) for t in want]
    at = [t.data_ptr() for t in got]
    if not twin:
        at[2] = at[3] = 0
    _lib.call("pt_quant_rowwise_colwise_rows_repeat", x.data_ptr(), rows, repeat, _lib.PT_BF16, M, H, H, index.data_ptr(), *at,
              _lib.PT_CH_TRANSPOSED, None, 0, _lib.stream_ptr(x.device))
    for i, (a, b) in enumerate(zip(got, want)):
        b = b.view(torch.uint8) if b.dtype == torch.float8_e4m3fn else b
        assert torch.equal(a, b if twin or i < 2 else torch.zeros_like(b))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,H,k,n", [(1, 8, 1, 0), (33, 264, 3, 1), (100, 2048, 6, 2), (7, 1024, 9, 3), (5, 12, 2, 2)])
def test_branch_gradients_are_summed_once(dtype, T, H, k, n):
    from pith_train_amd.operators.moe_combine import token_branches

    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn((T, H), generator=g, device="cuda").to(dtype).requires_grad_(True)
    rows, *others = token_branches(x, k, n)
    assert rows.shape == (T, k, H) and (k == 1 or rows.stride(1) == 0) and len(others) == n
    grads = [torch.randn(t.shape, generator=g, device="cuda").to(dtype) for t in (rows, *others)]
    for used in (slice(None), slice(0, 1), slice(1, None)):
        outs, gs = [rows, *others][used], grads[used]
        if not outs:
            continue
        (got,) = torch.autograd.grad(outs, x, gs, retain_graph=True)
        want = sum(t.double().sum(1) if t.dim() == 3 else t.double() for t in gs)
        tol = 2.0 ** -7 if dtype == torch.bfloat16 else 1e-5  # H = 12 takes torch's additions, each rounded
        assert ((got.double() - want).abs() <= tol * (want.abs() + 4)).all()
        if H % 8 == 0 and dtype == torch.bfloat16:
            assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()


@pytest.mark.parametrize("rows,hidden,width", [(1, 16, 128), (17, 144, 384), (129, 272, 128), (1000, 256, 640), (2049, 2048, 128), (4100, 512, 1408)])
def test_mlp_as_one_node(rows, hidden, width):
    """One row, ragged rows and widths, an input that is quantised with the weights and one that is not, split
    reductions: the result of the three linears, their weight gradients, and the input gradient up to the
    rounding of one addition; then again with the weights kept, and without a backward."""
    from pith_train_amd.modules import experts as X
    from pith_train_amd.operators.silu_mul import silu_mul

    g = torch.Generator().manual_seed(rows)
    mlp = X.DeepSeekV2MLP(hidden, width).cuda().to(torch.bfloat16)
    with torch.no_grad():
        for p in mlp.parameters():
            p.copy_((torch.randn(p.shape, generator=g) * 0.05).to(p.dtype))
    x = torch.randn((rows, hidden), generator=g).bfloat16().cuda().requires_grad_(True)
    dy = torch.randn((rows, hidden), generator=g).bfloat16().cuda()
    params = list(mlp.parameters())
    want = mlp.down_proj(silu_mul(mlp.gate_proj(x), mlp.up_proj(x)))
    want_grads = torch.autograd.grad(want, [x, *params], dy)
    for _ in range(2):  # weights quantised in the call, then kept
        got = mlp(x)
        grads = torch.autograd.grad(got, [x, *params], dy)
        assert got.grad_fn.name() != want.grad_fn.name()
        torch.testing.assert_close(got, want, rtol=0.01, atol=0.01 * want.float().abs().max().item())
        for a, b in zip(grads, want_grads):
            torch.testing.assert_close(a, b, rtol=0.01, atol=0.01 * b.float().abs().max().item())
    with torch.no_grad():
        assert torch.equal(mlp(x.view(1, rows, hidden))[0], got)


@pytest.mark.parametrize("family", ["Qwen3MoeExperts", "Qwen35MoeExperts", "GptOssExperts"])
def test_few_rows_whose_forward_turns_out_to_want_a_gradient(family):
    """Frozen experts on a few rows are handed groups of 64; behind a pre-hook that makes its rows require a gradient the
    forward keeps what the backward reads, in whole blocks of 128."""
    from pith_train_amd.modules import experts as X

    torch.manual_seed(5)
    m = getattr(X, family)(256, 128, 8).cuda().to(torch.bfloat16).requires_grad_(False)
    for p in m.parameters():
        p.normal_(0.0, 0.05)
    received = []

    def attach(module, args):
        received.append(args[0].detach().requires_grad_(True))
        return (received[-1], *args[1:])

    m.register_forward_pre_hook(attach)
    x = torch.randn((300, 256), device="cuda").bfloat16()
    idx, up = torch.randint(0, 7, (300,), device="cuda"), torch.randn((300, 256), device="cuda").bfloat16()
    out = X.forward_stage3(m, x, idx, 8)
    (grad,) = torch.autograd.grad(out, received[-1], up)
    m._forward_pre_hooks.clear()
    x.requires_grad_(True)
    want = X.forward_stage3(m, x, idx, 8)
    assert torch.equal(out, want) and torch.equal(grad, torch.autograd.grad(want, x, up)[0])
