"""GPU parity: the FP8 decompression of the MLA latent (kv_b) and its backward against the oracle's
dense FP8 linear (same quantised operands, fp64 accumulation), at DeepSeek-V2-Lite's shapes."""

import pytest
import torch

from oracle import gemm as G

pytestmark = pytest.mark.gpu


def _close(got, ref, what, rel=1e-2, diff=1e-3):
    got, ref = got.detach().float().cpu().double(), ref.double()
    assert got.shape == ref.shape, f"{what}: {tuple(got.shape)} vs {tuple(ref.shape)}"
    assert G.calc_diff(got, ref) < diff, what
    assert (got - ref).abs().max() <= rel * ref.abs().max() + 1e-30, what


@pytest.mark.parametrize("b,n,heads,nope,vdim,rank", [(1, 4096, 16, 128, 128, 512), (2, 384, 4, 64, 32, 256)])
def test_decompress_forward_backward(b, n, heads, nope, vdim, rank):
    from pith_train_amd.operators.deepgemm_quantize import fp8cast_blockwise_transpose
    from pith_train_amd.operators.mla_decompress import mla_decompress, mla_decompress_backward

    out_features = heads * (nope + vdim)
    g = torch.Generator().manual_seed(n)
    nkv = torch.randn((b, n, rank), generator=g).bfloat16()
    w = (torch.randn((out_features, rank), generator=g) * 0.02).bfloat16()
    dk = torch.randn((b, n, heads, nope), generator=g).bfloat16()
    dv = torch.randn((b, n, heads, vdim), generator=g).bfloat16()
    y_ref, saved = G.fp8_linear_forward(nkv.reshape(b * n, rank), w)
    dy = torch.cat([dk, dv], dim=-1).reshape(b * n, out_features)
    gi_ref, gw_ref = G.fp8_linear_backward(dy, saved)

    w_fp8, w_s, w_t_fp8, w_t_s = fp8cast_blockwise_transpose(w.cuda())
    k_nope, value = mla_decompress(nkv.cuda(), w.cuda(), heads, nope, vdim, use_fp8=True, weight_fp8=w_fp8, scale_weight=w_s)
    assert k_nope.shape == (b, n, heads, nope) and value.shape == (b, n, heads, vdim) and value.is_contiguous()
    kv_ref = y_ref.view(b, n, heads, nope + vdim)
    _close(k_nope, kv_ref[..., :nope], "k_nope")
    _close(value, kv_ref[..., nope:], "value")
    # the bf16 branch is the plain linear
    k2, v2 = mla_decompress(nkv.cuda(), w.cuda(), heads, nope, vdim)
    ref2 = torch.nn.functional.linear(nkv.cuda(), w.cuda()).view(b, n, heads, nope + vdim)
    assert torch.equal(k2, ref2[..., :nope]) and torch.equal(v2, ref2[..., nope:])

    d_nkv, dW = mla_decompress_backward(dk.cuda(), dv.cuda(), nkv.cuda(), w_t_fp8, w_t_s)
    assert d_nkv.dtype == torch.float32 and dW.dtype == torch.float32
    assert d_nkv.shape == (b, n, rank) and dW.shape == (out_features, rank)
    _close(d_nkv, gi_ref.view(b, n, rank), "d_nkv")
    _close(dW, gw_ref, "dW")


@pytest.mark.parametrize("rows,heads,nope,vdim,rank,fused", [
    (16, 1, 8, 8, 128, True), (129, 3, 24, 40, 144, True), (1000, 4, 64, 32, 256, True), (384, 4, 128, 128, 512, True),
    (520, 16, 128, 64, 512, True), (200, 2, 20, 44, 128, False)])
def test_per_head_halves_have_the_bits_of_the_concatenated_tensors(rows, heads, nope, vdim, rank, fused):
    """The GEMM that stores both halves of every head and the quantiser that reads them, against the dense
    linear on the concatenated tensors: ragged rows, widths below and across a tile's columns, and a
    width that is no multiple of 8, which goes the concatenated way."""
    from pith_train_amd.operators import linear as L
    from pith_train_amd.operators.deepgemm_quantize import fp8cast_blockwise_transpose, fp8cast_rowwise_blockwise_transpose
    from pith_train_amd.operators.mla_decompress import mla_decompress, mla_decompress_backward

    n = heads * (nope + vdim)
    g = torch.Generator().manual_seed(rows)
    x = torch.randn((rows, rank), generator=g).bfloat16().cuda()
    w_fp8, w_s, w_t, w_t_s = fp8cast_blockwise_transpose((torch.randn((n, rank), generator=g) * 0.02).bfloat16().cuda())
    dk = torch.randn((rows, heads, nope), generator=g).bfloat16().cuda()
    dv = torch.randn((rows, heads, vdim), generator=g).bfloat16().cuda()

    assert (L.fp8_act_weight_gemm_heads(x, w_fp8, w_s, heads, nope, vdim) is not None) == fused
    k_nope, value = mla_decompress(x[None], None, heads, nope, vdim, use_fp8=True, weight_fp8=w_fp8, scale_weight=w_s)
    kv = L.fp8_act_weight_gemm(x, w_fp8, w_s)[0].view(rows, heads, nope + vdim)
    assert torch.equal(k_nope[0], kv[..., :nope]) and torch.equal(value[0], kv[..., nope:])

    d_x, d_w = mla_decompress_backward(dk[None], dv[None], x[None], w_t, w_t_s)
    x_t, x_t_s = fp8cast_rowwise_blockwise_transpose(x, _padded=True)[2:]
    want = L.fp8_dgrad_wgrad(torch.cat([dk, dv], -1).view(rows, n), w_t, w_t_s, x_t, x_t_s, rank, _zero_padded=True)
    # the concatenated way rounds to bf16 before it widens
    assert torch.equal(d_x[0].bfloat16(), want[0]) and torch.equal(d_w.bfloat16(), want[1])


@pytest.mark.parametrize("rows,heads,nope,vdim,rank", [(1, 1, 8, 8, 16), (257, 3, 24, 40, 144), (8321, 2, 64, 72, 136)])
def test_gradients_and_latent_quantised_in_one_launch(rows, heads, nope, vdim, rank):
    """Against the two launches that it stands for: ragged tiles on every side, one tile, and row blocks in whole octets
    with some left over; the latent's rows lie in a wider buffer."""
    from pith_train_amd import _lib

    g = torch.Generator(device="cuda").manual_seed(rows)
    n, pitch, row_blocks = heads * (nope + vdim), (rows + 15) // 16 * 16 + 128, -(-rows // 128)

    def normal(*shape):
        return torch.randn(shape, device="cuda", generator=g).bfloat16()

    dk, dv, x = normal(rows, heads * nope), normal(rows, heads * vdim), normal(rows, rank + 8)
    results = []
    for together in (False, True):
        byte = lambda *s: torch.zeros(s, dtype=torch.uint8, device="cuda")  # noqa: E731
        q, q_t, x_t = byte(rows, n), byte(n, pitch), byte(rank, pitch)
        s, s_t, xs = (torch.zeros(z, device="cuda") for z in ((rows, -(-n // 128)), (n, row_blocks), (-(-rank // 128), row_blocks)))
        results.append((q, q_t, x_t, s, s_t, xs))
        grads = [_lib.ptr(dk), _lib.ptr(dv), rows, heads, nope, vdim, _lib.ptr(q), _lib.ptr(s), _lib.ptr(q_t), pitch, _lib.ptr(s_t)]
        if together:
            _lib.call("pt_quant_heads_and_input", *grads, _lib.ptr(x), rank, rank + 8, _lib.ptr(x_t), _lib.ptr(xs), _lib.stream_ptr())
        else:
            _lib.call("pt_quant_heads_rowwise_transpose_ld", *grads, _lib.stream_ptr())
            _lib.call("pt_quant_rowwise_blockwise_transpose_ld", _lib.ptr(x), _lib.PT_BF16, rows, rank, rank + 8, None, None, _lib.ptr(x_t), pitch, _lib.ptr(xs),
                      _lib.stream_ptr())
    assert all(torch.equal(a, b) for a, b in zip(*results)) and all(t.float().abs().sum() > 0 for t in results[0])
