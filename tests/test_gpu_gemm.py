"""GPU parity: FP8 GEMMs through the C-ABI vs the float64 dequantised oracle.

Tolerance (stated by the task): every element within 1e-2 relative of the fp32/fp64-dequantised
reference (with an absolute floor of 1e-2 x rms(ref) for elements near zero), and the reference
test-suite's similarity metric ``calc_diff < 1e-3``
(tests/test_deepgemm_fp8_linear_correctness.py:14,22-28).  In practice the only differences are
the fp32 accumulation order and the single bf16 rounding (2**-9).
"""

import pytest
import torch
from gemm_rules import schedule

from oracle import fp8 as Q
from oracle import gemm as G

pytestmark = pytest.mark.gpu

REL = 1e-2


@pytest.fixture(autouse=True, params=["auto", "p0", "q0", "q1", "r0", "t"])
def gemm_kernel(request):
    """Every test runs once per GEMM kernel of the library (and once with the library's own choice)."""
    from pith_train_amd import _lib

    _lib.call("pt_gemm_select_kernel", request.param.encode())
    yield request.param
    _lib.call("pt_gemm_select_kernel", None)


def _check(got, ref, what):
    got = got.float().cpu().double()
    ref = ref.double()
    assert got.shape == ref.shape
    assert torch.isfinite(got).all(), f"{what}: non-finite output"
    rms = ref.pow(2).mean().sqrt().item()
    err = (got - ref).abs()
    bound = REL * ref.abs() + REL * rms
    worst = (err - bound).max().item()
    assert worst <= 0, f"{what}: max violation {worst:.3e} (rms {rms:.3e}, max err {err.max().item():.3e})"
    assert G.calc_diff(got, ref) < 1e-3, f"{what}: calc_diff {G.calc_diff(got, ref):.3e}"


def _rand(shape, seed, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * std).bfloat16()


@pytest.mark.parametrize("M,N,K", [(128, 128, 128), (256, 384, 512), (1024, 512, 256), (300, 200, 384), (7, 128, 256),
                                   (512, 2880, 2880), (2048, 4096, 2048), (130, 64, 64)])
def test_dense_nt(M, N, K):
    from pith_train_amd.operators.linear import _fp8_gemm_nt

    x, w = _rand((M, K), M + K), _rand((N, K), N + K + 1, 0.02)
    a, sa, _, _ = Q.fp8cast_rowwise_transpose(x)
    b, sb, _, _ = Q.fp8cast_blockwise_transpose(w)
    ref = G.gemm_nt_dense(a, sa, b, sb, torch.float64)
    out = _fp8_gemm_nt(a.cuda(), sa.cuda(), b.cuda(), sb.cuda(), M, N, "cuda", torch.bfloat16)
    _check(out, ref, f"dense {M}x{N}x{K}")
    out32 = _fp8_gemm_nt(a.cuda(), sa.cuda(), b.cuda(), sb.cuda(), M, N, "cuda", torch.float32)
    _check(out32, ref, f"dense fp32 {M}x{N}x{K}")


@pytest.mark.parametrize("N", [1, 3, 4, 130, 259, 516])
def test_dense_nt_with_rows_that_are_no_whole_16_bytes(N):
    """Result rows that the 16-byte stores cannot write (as bf16, fp32 or both), ending inside a tile's first,
    second and third columns of blocks."""
    from pith_train_amd.operators.linear import _fp8_gemm_nt

    M, K = 300, 144
    a, sa, _, _ = Q.fp8cast_rowwise_transpose(_rand((M, K), N))
    b, sb, _, _ = Q.fp8cast_blockwise_transpose(_rand((N, K), N + 1, 0.02))
    ref = G.gemm_nt_dense(a, sa, b, sb, torch.float64)
    for dtype in (torch.bfloat16, torch.float32):
        _check(_fp8_gemm_nt(a.cuda(), sa.cuda(), b.cuda(), sb.cuda(), M, N, "cuda", dtype), ref, f"dense {M}x{N}x{K} {dtype}")


@pytest.mark.parametrize("M,N,K", [(512, 256, 4096), (300, 200, 4000), (128, 128, 20000), (256, 1024, 2048)])
def test_dense_nt_with_the_reduction_split_over_workgroups(M, N, K):
    """Small outputs with a long reduction (a dense weight gradient) are computed as several
    ranges of the reduction side by side and summed: same result within the GEMM tolerance, through
    the operator's own rule and through the C-ABI with other range lengths (ragged last range,
    one range)."""
    from pith_train_amd import _lib
    from pith_train_amd.operators.linear import _fp8_gemm_nt, _split_k

    x, w = _rand((M, K), M + K + 2), _rand((N, K), N + K + 3, 0.02)
    a, sa, _, _ = Q.fp8cast_rowwise_transpose(x)
    b, sb, _, _ = Q.fp8cast_blockwise_transpose(w)
    ref = G.gemm_nt_dense(a, sa, b, sb, torch.float64)
    assert _split_k(M, N, K)[0] > 1, "the case is meant to take the split path"
    ad, sad, bd, sbd = a.cuda(), sa.cuda(), b.cuda(), sb.cuda()
    _check(_fp8_gemm_nt(ad, sad, bd, sbd, M, N, "cuda", torch.bfloat16), ref, f"split dense {M}x{N}x{K}")
    for split_len in (128, 640, (K + 127) // 128 * 128):
        splits = (K + split_len - 1) // split_len
        partial = torch.full((splits, M, N), float("nan"), device="cuda")
        _lib.call("pt_gemm_nt_dense_splitk", ad.data_ptr(), sad.data_ptr(), bd.data_ptr(), sbd.data_ptr(), partial.data_ptr(),
                  splits, split_len, M, N, K, _lib.stream_ptr("cuda"))
        for dt in (torch.float32, torch.bfloat16):
            out = torch.empty((M, N), device="cuda", dtype=dt)
            _lib.call("pt_sum_partials", partial.data_ptr(), splits, M * N, out.data_ptr(), _lib.dtype_code(dt),
                      _lib.stream_ptr("cuda"))
            _check(out, ref, f"split dense {M}x{N}x{K} in {splits} ranges of {split_len} as {dt}")
        # the slabs are the partial products of their ranges: they add up in float64 as well
        _check(partial.double().sum(0), ref, "slabs")


def _dense_rows_against_oracle(M, N, K, rows, what):
    from pith_train_amd.operators.linear import _fp8_gemm_nt

    x, w = _rand((M, K), M + K + 4), _rand((N, K), N + K + 5, 0.02)
    a, sa, _, _ = Q.fp8cast_rowwise_transpose(x)
    b, sb, _, _ = Q.fp8cast_blockwise_transpose(w)
    out = _fp8_gemm_nt(a.cuda(), sa.cuda(), b.cuda(), sb.cuda(), M, N, "cuda", torch.bfloat16)
    assert out.shape == (M, N)
    ref = G.gemm_nt_dense(a[rows], sa[rows], b, sb, torch.float64)
    _check(out[rows.cuda()], ref, what)


def test_dense_nt_with_more_tiles_per_workgroup_than_the_tile_table_holds(gemm_kernel):
    """32768 x 25600 is 12800 tiles of 256 x 256, 50 per workgroup of the persistent kernels: the
    last tiles of every workgroup are decoded on the fly instead of read from the table built at
    kernel start.  Two rows of every 256-row tile are compared over all columns, so every tile of
    the launch is checked."""
    M, N, K = 32768, 25600, 128
    rows = torch.arange(0, M, 256).repeat_interleave(2) + torch.tensor([5, 201]).repeat(M // 256)
    _dense_rows_against_oracle(M, N, K, rows, f"dense {M}x{N}x{K}, {gemm_kernel}")


def test_dense_nt_with_an_output_beyond_the_32_bit_store_offsets(gemm_kernel):
    """A 65536 x 32896 bf16 result is 4.3 GB: past the unsigned 32-bit byte offsets the persistent
    kernels store through, so the library must route the call to its kernel with 64-bit addresses
    whatever kernel was asked for.  One row of every 128-row tile, all columns."""
    if gemm_kernel not in ("auto", "q0"):
        pytest.skip("the route does not depend on the requested kernel; run twice")
    M, N, K = 65536, 32896, 128
    assert M * N * 2 >= 1 << 32
    rows = torch.arange(0, M, 128) + (torch.arange(M // 128) * 37) % 128
    _dense_rows_against_oracle(M, N, K, rows, f"dense {M}x{N}x{K} (64-bit route)")


def test_dense_scale_extremes():
    """Rows with very different magnitudes: the E8M0 exponents given to the MFMA must be per row."""
    from pith_train_amd.operators.linear import _fp8_gemm_nt

    M, N, K = 256, 256, 512
    g = torch.Generator().manual_seed(5)
    x = (torch.randn((M, K), generator=g) * torch.exp2(torch.randint(-20, 20, (M, 1), generator=g).float())).bfloat16()
    w = (torch.randn((N, K), generator=g) * torch.exp2(torch.randint(-10, 10, (N // 128, 1), generator=g).float())
         .repeat_interleave(128, 0)).bfloat16()
    a, sa, _, _ = Q.fp8cast_rowwise_transpose(x)
    b, sb, _, _ = Q.fp8cast_blockwise_transpose(w)
    ref = G.gemm_nt_dense(a, sa, b, sb, torch.float64)
    out = _fp8_gemm_nt(a.cuda(), sa.cuda(), b.cuda(), sb.cuda(), M, N, "cuda", torch.float32).cpu().double()
    # compare row by row relative to each row's own scale
    rel = (out - ref).abs().amax(1) / ref.abs().amax(1).clamp_min(1e-300)
    assert rel.max().item() < 1e-4, rel.max().item()


def _groups(sizes):
    ks = torch.tensor([(s + 127) // 128 * 128 for s in sizes], dtype=torch.int32)
    return ks, ks.cumsum(0).to(torch.int32)


GROUPED = [
    ([128, 128], 256, 128),
    ([100, 0, 300, 128, 1], 512, 256),
    ([0, 0, 640], 384, 384),
    ([256] * 8, 512, 256),
    ([512, 640, 128, 0, 384], 1536, 2048),
    ([300, 200], 2880, 2880),
    ([1536, 1700], 256, 2048),  # large groups + long reduction: the pipelined loop by the library's own choice
]


# More than 256 groups: the kernels' group scan gives every lane more than four groups (its long
# path), and the list of tiles is full of empty and single-block groups.
MANY_GROUPS = [([0 if i % 7 == 3 else (256 if i % 5 == 0 else 128) for i in range(320)], 256, 256)]


@pytest.mark.parametrize("sizes,N,K", GROUPED + MANY_GROUPS)
def test_m_grouped_nt(sizes, N, K):
    from pith_train_amd.operators.grouped_linear import m_grouped_fp8_gemm_nt

    ks, offs = _groups(sizes)
    M, Gn = int(offs[-1]), len(sizes)
    x = _rand((M, K), M + K)
    start = 0
    for s, k in zip(sizes, ks.tolist()):  # zero pad rows like the scatter does
        x[start + s : start + k] = 0
        start += k
    w = _rand((Gn, N, K), N + K + 3, 0.02)
    a, sa, _, _ = Q.fp8cast_rowwise_colwise(x)
    b, sb, _, _ = Q.fp8cast_blockwise_transpose_batched(w)
    ref = G.gemm_m_grouped_nt(a, sa, b, sb, offs, torch.float64)
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    m_grouped_fp8_gemm_nt((a.cuda(), sa.cuda()), (b.cuda(), sb.cuda()), out, offs.cuda())
    _check(out, ref, f"m-grouped {sizes} N={N} K={K}")


@pytest.mark.parametrize("sizes,N,K", GROUPED)
def test_m_grouped_nt_scattered_rows(sizes, N, K, gemm_kernel):
    """The un-permute folded into the store: result row r lands in output row out_rows[r]; rows of
    a group's padding (negative index) are dropped and rows nobody maps to stay untouched."""
    from pith_train_amd.operators.grouped_linear import m_grouped_fp8_gemm_nt

    if gemm_kernel == "t":
        pytest.skip("the tile-per-workgroup kernel has no scattered store (the library refuses it)")
    ks, offs = _groups(sizes)
    M, Gn = int(offs[-1]), len(sizes)
    x = _rand((M, K), M + K + 17)
    w = _rand((Gn, N, K), N + K + 5, 0.02)
    a, sa, _, _ = Q.fp8cast_rowwise_colwise(x)
    b, sb, _, _ = Q.fp8cast_blockwise_transpose_batched(w)
    ref = G.gemm_m_grouped_nt(a, sa, b, sb, offs, torch.float64)
    real = torch.zeros(M, dtype=torch.bool)
    start = 0
    for s_, k_ in zip(sizes, ks.tolist()):
        real[start : start + s_] = True
        start += k_
    n_real = int(real.sum())
    out_m = n_real + 3  # three rows that no result row maps to
    g = torch.Generator().manual_seed(M)
    dst = torch.randperm(out_m, generator=g)[:n_real].to(torch.int32)
    out_rows = torch.full((M,), -1, dtype=torch.int32)
    out_rows[real] = dst
    out = torch.full((out_m, N), 7.0, dtype=torch.bfloat16, device="cuda")
    m_grouped_fp8_gemm_nt((a.cuda(), sa.cuda()), (b.cuda(), sb.cuda()), out, offs.cuda(), out_rows.cuda())
    out = out.cpu()
    _check(out[dst.long()], ref[real], f"m-grouped scattered {sizes} N={N} K={K}")
    untouched = torch.ones(out_m, dtype=torch.bool)
    untouched[dst.long()] = False
    assert (out[untouched] == 7.0).all()


@pytest.mark.parametrize("sizes,N,K", GROUPED + MANY_GROUPS + [([256], 272, 400), ([600] * 16, 768, 2048)])
def test_m_grouped_nn_reads_the_forward_layout_weight_with_the_bits_of_nt(sizes, N, K, gemm_kernel):
    """The input-gradient form: b given reduction-major ([G, K, N], scales [G, K/128, N/128]) is the
    same product as the NT form on its transpose, accumulated in the same order: equal to the
    oracle within the GEMM tolerance and to the NT kernel bit for bit, plain and with scattered
    rows, for ragged N and K too."""
    from pith_train_amd.operators.grouped_linear import m_grouped_fp8_gemm_nn, m_grouped_fp8_gemm_nt

    ks, offs = _groups(sizes)
    M, Gn = int(offs[-1]), len(sizes)
    x = _rand((M, K), M + K + 29)
    w = _rand((Gn, N, K), N + K + 31, 0.02)
    a, sa, _, _ = Q.fp8cast_rowwise_colwise(x)
    b, sb, _, _ = Q.fp8cast_blockwise_transpose_batched(w)
    ref = G.gemm_m_grouped_nt(a, sa, b, sb, offs, torch.float64)
    bt, sbt = b.transpose(1, 2).contiguous().cuda(), sb.transpose(1, 2).contiguous().cuda()
    out_nn = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    out_nt = out_nn.clone()
    m_grouped_fp8_gemm_nn((a.cuda(), sa.cuda()), (bt, sbt), out_nn, offs.cuda())
    _check(out_nn, ref, f"m-grouped nn {sizes} N={N} K={K}")
    if gemm_kernel in ("auto", "r0"):  # the NT launch of the same kernel family
        m_grouped_fp8_gemm_nt((a.cuda(), sa.cuda()), (b.cuda(), sb.cuda()), out_nt, offs.cuda())
        assert torch.equal(out_nn[: int(offs[-1])], out_nt[: int(offs[-1])])
    if N % 8 == 0:
        g = torch.Generator().manual_seed(M + 1)
        dst = torch.randperm(M + 5, generator=g)[:M].to(torch.int32)
        dst[::7] = -1  # dropped rows
        out_s = torch.full((M + 5, N), 7.0, dtype=torch.bfloat16, device="cuda")
        m_grouped_fp8_gemm_nn((a.cuda(), sa.cuda()), (bt, sbt), out_s, offs.cuda(), dst.cuda())
        keep = (dst >= 0).nonzero().flatten()
        assert torch.equal(out_s[dst[keep].long().cuda()], out_nn[keep.cuda()])
        untouched = torch.ones(M + 5, dtype=torch.bool)
        untouched[dst[keep].long()] = False
        assert (out_s.cpu()[untouched] == 7.0).all()


@pytest.mark.parametrize("sizes", [[256], [256, 384]])
def test_m_grouped_nn_reads_nothing_past_a_ragged_reduction(sizes):
    """The reduction-major b operand of a ragged reduction (K = 400: 16 rows into the last
    128-block) lies inside a larger buffer whose every other byte is 0xFF, an e4m3 NaN: the rows of
    a reduction block past a group's K rows belong to the next group or to that padding, and the
    loader leaves them to the range check of the group's buffer descriptor.  A byte read from
    there would meet a zero of the a operand and give NaN; the result must be finite and equal to
    the NT form's bit for bit."""
    from pith_train_amd.operators.grouped_linear import m_grouped_fp8_gemm_nn, m_grouped_fp8_gemm_nt

    N, K = 272, 400
    ks, offs = _groups(sizes)
    M, Gn = int(offs[-1]), len(sizes)
    x = _rand((M, K), 71)
    w = _rand((Gn, N, K), 73, 0.02)
    a, sa, _, _ = Q.fp8cast_rowwise_colwise(x)
    b, sb, _, _ = Q.fp8cast_blockwise_transpose_batched(w)
    big = torch.full((Gn * K * N + 256 * N,), 0xFF, dtype=torch.uint8, device="cuda")
    bt = big[: Gn * K * N].view(Gn, K, N)
    bt.copy_(b.transpose(1, 2).contiguous().view(torch.uint8).cuda())
    bt = bt.view(torch.float8_e4m3fn)
    sbt = sb.transpose(1, 2).contiguous().cuda()
    out_nn = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    out_nt = out_nn.clone()
    m_grouped_fp8_gemm_nn((a.cuda(), sa.cuda()), (bt, sbt), out_nn, offs.cuda())
    m_grouped_fp8_gemm_nt((a.cuda(), sa.cuda()), (b.cuda(), sb.cuda()), out_nt, offs.cuda())
    rows = int(offs[-1])
    assert torch.isfinite(out_nn[:rows].float()).all(), "a byte past the group's reduction rows was read"
    assert torch.equal(out_nn[:rows], out_nt[:rows])
    assert (big[Gn * K * N :] == 0xFF).all()


def test_m_grouped_nt_with_more_tiles_per_workgroup_than_the_tile_table_holds(gemm_kernel):
    """Four groups of 25600 rows x 8192 columns: 12800 tiles, 50 per workgroup, so the grouped
    tile decode (group search, row tile inside the group) also runs on the fly for the last tiles.
    Two rows of every 256-row tile against the oracle, all columns."""
    from pith_train_amd.operators.grouped_linear import m_grouped_fp8_gemm_nt

    sizes, N, K = [25600] * 4, 8192, 128
    ks, offs = _groups(sizes)
    M, Gn = int(offs[-1]), len(sizes)
    x, w = _rand((M, K), M + K + 6), _rand((Gn, N, K), N + K + 7, 0.02)
    a, sa, _, _ = Q.fp8cast_rowwise_colwise(x)
    b, sb, _, _ = Q.fp8cast_blockwise_transpose_batched(w)
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    m_grouped_fp8_gemm_nt((a.cuda(), sa.cuda()), (b.cuda(), sb.cuda()), out, offs.cuda())
    rows = torch.arange(0, M, 256).repeat_interleave(2) + torch.tensor([9, 250]).repeat(M // 256)
    grp = rows // 25600
    for g in range(Gn):
        r = rows[grp == g]
        ref = G.gemm_nt_dense(a[r], sa[r], b[g], sb[g], torch.float64)
        _check(out[r.cuda()], ref, f"m-grouped group {g} of {sizes} N={N} K={K}, {gemm_kernel}")


def test_k_grouped_wgrad_with_more_tiles_per_workgroup_than_the_tile_table_holds(gemm_kernel):
    """200 groups of one 128-row block, 2048 x 2048 results: 12800 tiles, 50 per workgroup.  Groups
    spread over the whole list (the on-the-fly decode handles the end of every XCD's share) are
    compared with the oracle; all others must at least be finite and non-trivial."""
    from pith_train_amd.operators.grouped_linear import k_grouped_fp8_wgrad

    if gemm_kernel == "t":
        pytest.skip("the tile-per-workgroup kernel has no tile table")
    Gn, N, K = 200, 2048, 2048
    ks, offs = _groups([128] * Gn)
    M = int(offs[-1])
    dy, x = _rand((M, N), M + N + 1), _rand((M, K), M + K + 2)
    _, _, dy_ch, dy_s = Q.fp8cast_rowwise_colwise(dy)
    _, _, x_ch, x_s = Q.fp8cast_rowwise_colwise(x)
    tr = lambda q: q.view(torch.uint8).T.contiguous().view(torch.float8_e4m3fn).cuda()  # noqa: E731
    out = torch.full((Gn, N, K), float("nan"), dtype=torch.bfloat16, device="cuda")
    k_grouped_fp8_wgrad((tr(dy_ch), dy_s.cuda()), (tr(x_ch), x_s.cuda()), out, offs.cuda(), False)
    assert torch.isfinite(out).all()
    assert (out.float().abs().amax(dim=(1, 2)) > 0).all()
    for g in list(range(23, Gn, 25)) + [0, Gn - 1]:  # 24, 49, ..., 199: the last group of every eighth of the list
        sl = slice(g * 128, (g + 1) * 128)
        ref = G.gemm_k_grouped_wgrad(dy_ch[sl], dy_s[g : g + 1], x_ch[sl], x_s[g : g + 1], torch.tensor([128], dtype=torch.int32), 1,
                                     torch.float64).double()
        _check(out[g : g + 1], ref, f"wgrad group {g} of {Gn}, {gemm_kernel}")


# Skewed group sizes: the weight-gradient tiles are shared out over the XCDs by cost (a tile's
# reduction length), so the cuts fall inside groups, at empty groups and at the ends of the list.
SKEWED = [
    ([0] * 5 + [4096] + [0] * 10 + [130, 1, 1, 1], 512, 512),
    ([3, 900, 0, 17, 2500, 128, 0, 0, 1, 640] * 7, 256, 256),
    ([2000], 768, 256),
    ([1] * 9, 256, 512),
]


@pytest.mark.parametrize("sizes,N,K", GROUPED + SKEWED + MANY_GROUPS)
@pytest.mark.parametrize("accumulate", [False, True])
def test_k_grouped_wgrad(sizes, N, K, accumulate):
    from pith_train_amd.operators.grouped_linear import k_grouped_fp8_wgrad

    if N * K > 4e6 and accumulate:
        pytest.skip("covered by the non-accumulating case")
    ks, offs = _groups(sizes)
    M, Gn = int(offs[-1]), len(sizes)
    dy, x = _rand((M, N), M + N), _rand((M, K), M + K + 9)
    _, _, dy_ch, dy_s = Q.fp8cast_rowwise_colwise(dy)
    _, _, x_ch, x_s = Q.fp8cast_rowwise_colwise(x)
    ref = G.gemm_k_grouped_wgrad(dy_ch, dy_s, x_ch, x_s, offs, Gn, torch.float64).double()
    tr = lambda q: q.view(torch.uint8).T.contiguous().view(torch.float8_e4m3fn).cuda()  # noqa: E731
    a, b = (tr(dy_ch), dy_s.cuda()), (tr(x_ch), x_s.cuda())
    if not accumulate:
        out = torch.full((Gn, N, K), float("nan"), dtype=torch.bfloat16, device="cuda")
        k_grouped_fp8_wgrad(a, b, out, offs.cuda(), False)
        _check(out, ref, "wgrad bf16")
        out32 = torch.full((Gn, N, K), float("nan"), dtype=torch.float32, device="cuda")
        k_grouped_fp8_wgrad(a, b, out32, offs.cuda(), False)
        _check(out32, ref, "wgrad fp32")
        for g, s in enumerate(sizes):
            if s == 0:
                assert (out[g] == 0).all(), "empty group must give exactly zero"
    else:
        old = _rand((Gn, N, K), 77, 30.0)
        out = old.clone().cuda()
        k_grouped_fp8_wgrad(a, b, out, offs.cuda(), True)
        # bf16(old + bf16(sum)): same two roundings as `weight.grad += wgrad.to(bf16)`
        expect = (old.float() + ref.float().bfloat16().float()).bfloat16()
        diff = (out.cpu().float() - expect.float()).abs()
        # one bf16 ulp of slack: the kernel's fp32 sum may round to the neighbouring bf16 value
        # (relative to the operands, not to the possibly cancelling result)
        # plus the fp32 accumulation-order noise of the sum itself (matters where it cancels to ~0)
        ulp = (old.float().abs() + ref.float().abs()) * 2.0**-6 + 1e-3 * ref.float().pow(2).mean().sqrt()
        assert (diff <= ulp).all(), diff.max().item()
        old32 = old.float()
        out32 = old32.clone().cuda()
        k_grouped_fp8_wgrad(a, b, out32, offs.cuda(), True)
        _check(out32.cpu().double() - old32.double(), ref, "wgrad fp32 accumulate")


def test_k_grouped_wgrad_on_column_slices_of_the_scale_array():
    """The weight gradient of one half of a fused projection: rows of the transposed bytes (contiguous)
    and a column slice of the scale array (its row stride is passed to the library)."""
    from pith_train_amd.operators.grouped_linear import k_grouped_fp8_wgrad

    sizes, N, K = [300, 0, 200, 128], 256, 128
    ks, offs = _groups(sizes)
    M, Gn = int(offs[-1]), len(sizes)
    dy, x = _rand((M, N), 31), _rand((M, K), 32)
    _, _, dy_ch, dy_s = Q.fp8cast_rowwise_colwise(dy)
    _, _, x_ch, x_s = Q.fp8cast_rowwise_colwise(x)
    tr = lambda q: q.view(torch.uint8).T.contiguous().view(torch.float8_e4m3fn).cuda()  # noqa: E731
    dy_t, dy_sc, x_t, x_sc = tr(dy_ch), dy_s.cuda(), tr(x_ch), x_s.cuda()
    half = N // 2
    for lo in (0, half):
        ref = G.gemm_k_grouped_wgrad(dy_ch[:, lo : lo + half].contiguous(), dy_s[:, lo : lo + half].contiguous(), x_ch, x_s,
                                     offs, Gn, torch.float64).double()
        out = torch.full((Gn, half, K), float("nan"), dtype=torch.bfloat16, device="cuda")
        k_grouped_fp8_wgrad((dy_t[lo : lo + half], dy_sc[:, lo : lo + half]), (x_t, x_sc), out, offs.cuda(), False)
        _check(out, ref, f"wgrad on scale columns {lo}..{lo + half}")


@pytest.mark.parametrize("K", [128, 144, 256, 400])
@pytest.mark.parametrize("sizes,N", [([128, 0, 384, 250], 8), ([300, 128], 264), ([640, 1], 520)])
def test_m_grouped_scattered_rows_with_bias_of_short_reductions(sizes, N, K, gemm_kernel):
    """Output rows and bias of a tile are fetched during its first reduction block, which here is the
    only one or one of two to four; tiles end inside the columns.  Same bits as adding the bias to the
    plain result and moving the rows."""
    from pith_train_amd import _lib

    if gemm_kernel == "t":
        pytest.skip("the tile-per-workgroup kernel has no scattered store (the library refuses it)")
    ks, offs = _groups(sizes)
    M, Gn = int(offs[-1]), len(sizes)
    a, sa, _, _ = Q.fp8cast_rowwise_colwise(_rand((M, K), M + K))
    b, sb, _, _ = Q.fp8cast_blockwise_transpose_batched(_rand((Gn, N, K), N + K, 0.02))
    a, sa, b, sb, offs, bias = a.cuda(), sa.cuda(), b.cuda(), sb.cuda(), offs.cuda(), _rand((Gn, N), K).cuda()
    rows = torch.randperm(M, generator=torch.Generator().manual_seed(K)).int().cuda()
    plain, out = (torch.empty((M, N), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    args = [_lib.ptr(a), _lib.ptr(sa), _lib.ptr(b), _lib.ptr(sb)]
    dims = [_lib.dtype_code(torch.bfloat16), _lib.ptr(offs), Gn, M, N, K]
    _lib.call("pt_gemm_m_grouped_nt", *args, _lib.ptr(plain), *dims, _lib.stream_ptr())
    _lib.call("pt_gemm_m_grouped_nt_scatter_bias", *args, _lib.ptr(out), *dims, _lib.ptr(rows), M, _lib.ptr(bias), _lib.stream_ptr())
    group = torch.repeat_interleave(torch.arange(Gn, device="cuda"), torch.diff(offs, prepend=offs.new_zeros(1)).long())
    assert torch.equal(out[rows.long()], plain + bias[group])


@pytest.mark.parametrize("groups,N,W", [(3, 1024, 2048), (40, 1100, 1800), (256, 1024, 1280)])
def test_k_grouped_schedule_of_skewed_groups(gemm_kernel, groups, N, W):
    """A group of half of the rows, two of a quarter and so on, the others small or empty, so that workgroups are dealt the
    big tiles one by one: every tile is computed, once (accumulating), with the bits of the kernel that takes one small
    tile per workgroup."""
    from pith_train_amd import _lib

    if gemm_kernel != "auto":
        pytest.skip("the test selects the kernels itself; run once")
    g = torch.Generator(device="cuda").manual_seed(groups)
    tiles = -(-N // 256) * -(-W // 256)
    total = 1.3 * 96 * 256 / tiles  # blocks: a share of 125
    blocks = torch.randint(0, 3, (groups,), generator=torch.Generator().manual_seed(groups))
    for i, share in enumerate((2, 4, 4, 8, 8, 16, 32)[:groups]):
        blocks[i * (groups // 7 or 1)] = int(total / share)
    offs, M = torch.cumsum(blocks * 128, 0).int().cuda(), int(blocks.sum()) * 128
    assert schedule(blocks.tolist(), tiles, min(256, groups * tiles))[0] == "parts"

    def fp8(*shape):
        return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g) & 0xBF  # finite values below 2

    def scale(*shape):
        return torch.exp2(torch.randint(-6, 3, shape, device="cuda", generator=g).float())

    d, sd, x, sx = fp8(N, M), scale(M // 128, N), fp8(W, M), scale(M // 128, W)
    start = torch.randn((groups, N, W), device="cuda", generator=g).bfloat16()
    for add in (0, 1):
        out = []
        for kernel in (b"r0", b"s128"):
            _lib.call("pt_gemm_select_kernel", kernel)
            o = start.clone()
            _lib.call("pt_gemm_k_grouped_wgrad", _lib.ptr(d), _lib.ptr(sd), _lib.ptr(x), _lib.ptr(sx), _lib.ptr(o), _lib.dtype_code(o.dtype), add,
                      _lib.ptr(offs), groups, M, N, W, _lib.stream_ptr())
            out.append(o)
        assert torch.equal(*out)


@pytest.mark.parametrize("N,K", [(256, 128), (272, 1408), (2880, 2880)])
def test_row_scales_by_block(gemm_kernel, N, K):
    """The quantiser writes the same scales as [K/128, M], and every grouped GEMM that reads them so has the bits of
    the one that reads [M, K/128]: tiles past the last row and column, a reduction that ends inside a block."""
    from pith_train_amd import _lib

    g = torch.Generator(device="cuda").manual_seed(K)
    rows = torch.tensor([128, 0, 384, 640], dtype=torch.int32)
    G_, M, KB = len(rows), int(rows.sum()), (K + 127) // 128
    offs = torch.cumsum(rows, 0).int().cuda()
    x = torch.randn((M, K), device="cuda", generator=g).bfloat16() * torch.exp2(torch.randint(-9, 9, (M, 1), device="cuda", generator=g).float()).bfloat16()
    q, q2 = (torch.empty((M, K), dtype=torch.uint8, device="cuda") for _ in range(2))
    t, t2 = (torch.empty((K, M), dtype=torch.uint8, device="cuda") for _ in range(2))
    s, s2 = torch.empty((M, KB), device="cuda"), torch.empty((KB, M), device="cuda")
    ts, ts2 = (torch.empty((M // 128, K), device="cuda") for _ in range(2))
    bf16 = _lib.dtype_code(torch.bfloat16)
    _lib.call("pt_quant_rowwise_colwise", _lib.ptr(x), bf16, M, K, K, _lib.ptr(q), _lib.ptr(s), _lib.ptr(t), _lib.ptr(ts), _lib.PT_CH_TRANSPOSED, None, 0,
              _lib.stream_ptr())
    _lib.call("pt_quant_rowwise_colwise_by_block", _lib.ptr(x), bf16, M, K, K, _lib.ptr(q2), _lib.ptr(s2), _lib.ptr(t2), _lib.ptr(ts2), _lib.stream_ptr())
    assert torch.equal(q, q2) and torch.equal(t, t2) and torch.equal(ts, ts2) and torch.equal(s, s2.t())
    b = torch.randint(0, 256, (G_, N, K), dtype=torch.uint8, device="cuda", generator=g) & 0xBF
    b_s = torch.exp2(torch.randint(-6, 3, (G_, (N + 127) // 128, KB), device="cuda", generator=g).float())
    b_t, b_ts = b.transpose(1, 2).contiguous(), b_s.transpose(1, 2).contiguous()
    to = torch.randperm(M, device="cuda", generator=g).int()
    for reduction_major, scatter in ((0, False), (0, True), (1, False), (1, True)):
        if gemm_kernel == "t" and scatter and not reduction_major:
            continue  # refused: that kernel stores no scattered rows
        w, w_s = (b_t, b_ts) if reduction_major else (b, b_s)
        want, got = (torch.zeros((M, N), dtype=torch.bfloat16, device="cuda") for _ in range(2))
        name = "pt_gemm_m_grouped_" + ("nn" if reduction_major else "nt") + ("_scatter" if scatter else "")
        _lib.call(name, _lib.ptr(q), _lib.ptr(s), _lib.ptr(w), _lib.ptr(w_s), _lib.ptr(want), bf16, _lib.ptr(offs), G_, M, N, K,
                  *((_lib.ptr(to), M) if scatter else ()), _lib.stream_ptr())
        _lib.call("pt_gemm_m_grouped_by_block", _lib.ptr(q), _lib.ptr(s2), _lib.ptr(w), _lib.ptr(w_s), reduction_major, _lib.ptr(got), bf16, _lib.ptr(offs),
                  G_, M, N, K, _lib.ptr(to) if scatter else None, M if scatter else 0, _lib.stream_ptr())
        assert torch.equal(want, got)


@pytest.mark.parametrize("users", ["one", "some", "many", "outside"])
@pytest.mark.parametrize("N,K", [(256, 128), (272, 272), (2880, 1408)])
def test_rows_of_two_outputs(gemm_kernel, N, K, users):
    """An input gradient whose rows are summed by the row they expand: stored to the sum's place where there is nothing
    to add, and summed from a second output elsewhere, against scattering all of it and summing all of it.  Every
    source row used once, some not at all and some by two, one by more than a wave's lanes, indices outside the rows."""
    from pith_train_amd import _lib

    if gemm_kernel in ("p0", "q0", "q1", "t"):
        pytest.skip("names of r0, and a kernel that stores no scattered rows")
    g = torch.Generator(device="cuda").manual_seed(N + K)
    rows = torch.tensor([128, 0, 384, 640], dtype=torch.int32)
    G_, M, KB = len(rows), int(rows.sum()), (K + 127) // 128
    offs = torch.cumsum(rows, 0).int().cuda()
    n = M - 200  # rows of padding among the grouped ones
    row_map = torch.full((M,), -1, dtype=torch.int32, device="cuda")
    row_map[torch.randperm(M, device="cuda", generator=g)[:n]] = torch.randperm(n, device="cuda", generator=g).int()
    src = {"one": n, "some": n, "many": 40, "outside": n // 2}[users]
    index = torch.randperm(n, device="cuda", generator=g) if users == "one" else torch.randint(0, src, (n,), device="cuda", generator=g)
    if users == "many":
        index[: n // 2] = 7
    if users == "outside":
        index[::5] = src
        index[1::7] = -1
    q = torch.randint(0, 256, (M, K), dtype=torch.uint8, device="cuda", generator=g) & 0xBF
    q_s = torch.exp2(torch.randint(-6, 3, (KB, M), device="cuda", generator=g).float())
    b = torch.randint(0, 256, (G_, N, K), dtype=torch.uint8, device="cuda", generator=g) & 0xBF
    b_s = torch.exp2(torch.randint(-6, 3, (G_, (N + 127) // 128, KB), device="cuda", generator=g).float())
    bf16, stream = _lib.dtype_code(torch.bfloat16), _lib.stream_ptr()
    size = _lib.query("pt_gather_rows_backward_workspace_bytes", n, src)
    ws, dest = torch.empty(size, dtype=torch.uint8, device="cuda"), torch.empty(M, dtype=torch.int32, device="cuda")
    for reduction_major in (0, 1):
        w, w_s = (b.transpose(1, 2).contiguous(), b_s.transpose(1, 2).contiguous()) if reduction_major else (b, b_s)
        all_rows, shared = (torch.full((n, N), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
        want, got = (torch.full((src, N), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
        operands = (_lib.ptr(q), _lib.ptr(q_s), _lib.ptr(w), _lib.ptr(w_s), reduction_major)
        _lib.call("pt_gemm_m_grouped_by_block", *operands, _lib.ptr(all_rows), bf16, _lib.ptr(offs), G_, M, N, K, _lib.ptr(row_map), n, stream)
        _lib.call("pt_gather_rows_backward", _lib.ptr(all_rows), N, _lib.ptr(want), N, _lib.ptr(index), n, src, N, bf16, _lib.ptr(ws), size, stream)
        _lib.call("pt_gather_rows_backward_begin", _lib.ptr(index), n, src, _lib.ptr(ws), size, _lib.ptr(row_map), _lib.ptr(dest), M, stream)
        _lib.call("pt_gemm_m_grouped_by_block_two", *operands, _lib.ptr(got), _lib.ptr(shared), bf16, _lib.ptr(offs), G_, M, N, K, _lib.ptr(dest), src, n,
                  stream)
        _lib.call("pt_gather_rows_backward_shared", _lib.ptr(shared), N, _lib.ptr(got), N, n, src, N, bf16, _lib.ptr(ws), size, stream)
        assert torch.isfinite(want.float()).all() and torch.equal(got, want)


@pytest.mark.parametrize("reduction_major", [0, 1])
@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("N,K", [(528, 272), (768, 1408), (272, 2064)])
def test_ends_of_many_groups(gemm_kernel, N, K, two, reduction_major):
    """From 64 groups on the kernel of large tiles ends a group at its last used row, as the one of small tiles always does:
    groups that end 1, 7, 8, 9, 64, 65, 127 and 128 rows into their last block, of one to three blocks, and empty ones, stored
    to one output and to two.  The bits of a launch whose rows all count, nothing else written, whatever padding holds."""
    from pith_train_amd import _lib

    if gemm_kernel in ("p0", "q0", "q1", "t"):
        pytest.skip("names of r0, and a kernel that stores no scattered rows")
    g = torch.Generator(device="cuda").manual_seed(N + K)
    G_, KB = 66, (K + 127) // 128
    ends = [(1, 7, 8, 9, 64, 65, 127, 128)[i % 8] for i in range(G_)]
    blocks = [0 if i % 11 == 5 else 1 + i % 3 for i in range(G_)]
    rows = torch.tensor(blocks, dtype=torch.int32) * 128
    M = int(rows.sum())
    offs = torch.cumsum(rows, 0).int().cuda()
    used = torch.cat([(torch.arange(128 * b) < 128 * (b - 1) + e) for b, e in zip(blocks, ends)]).cuda()
    q = torch.randint(0, 256, (M, K), dtype=torch.uint8, device="cuda", generator=g) & 0xBF
    q_s = torch.exp2(torch.randint(-6, 3, (KB, M), device="cuda", generator=g).float())
    b = torch.randint(0, 256, (G_, K, N) if reduction_major else (G_, N, K), dtype=torch.uint8, device="cuda", generator=g) & 0xBF
    b_s = torch.exp2(torch.randint(-6, 3, (G_, KB, (N + 127) // 128) if reduction_major else (G_, (N + 127) // 128, KB), device="cuda", generator=g).float())
    to = torch.randperm(M, device="cuda", generator=g).int()
    second = torch.rand(M, device="cuda", generator=g) < 0.5

    def run(counts, a, a_s):
        index = torch.where(counts, torch.where(second, -2 - to, to) if two else to, -1).int()
        outs = [torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
        args = [_lib.ptr(a), _lib.ptr(a_s), _lib.ptr(b), _lib.ptr(b_s), reduction_major, _lib.ptr(outs[0])]
        sizes = [_lib.dtype_code(torch.bfloat16), _lib.ptr(offs), G_, M, N, K, _lib.ptr(index), M]
        if two:
            _lib.call("pt_gemm_m_grouped_by_block_two", *args, _lib.ptr(outs[1]), *sizes, M, _lib.stream_ptr())
        else:
            _lib.call("pt_gemm_m_grouped_by_block", *args, *sizes, _lib.stream_ptr())
        return outs

    want = run(torch.ones_like(used), q, q_s)
    dirty, dirty_s = q.clone(), q_s.clone()
    dirty[~used] = 0x7F  # not a number
    dirty_s[:, ~used] = float("nan")
    got = run(used, dirty, dirty_s)
    for i in range(2):
        mine = used & (second == bool(i)) if two else used if i == 0 else torch.zeros_like(used)
        place = to[mine].long()
        assert torch.isfinite(want[i][place].float()).all() and torch.equal(got[i][place], want[i][place])
        rest = torch.ones(M, dtype=torch.bool, device="cuda")
        rest[place] = False
        assert got[i][rest].isnan().all()


@pytest.mark.parametrize("tiles", [1, 3, 4, 10])
def test_grouped_tile_order_at_the_edges_of_its_strips(gemm_kernel, tiles):
    """Groups with more row tiles than column tiles and the other way round, one strip and several of unequal
    width, empty groups among them: the bits of the kernel that takes one small tile per workgroup, whatever
    place the order gives a tile."""
    from pith_train_amd import _lib

    if gemm_kernel != "auto":
        pytest.skip("the test selects the kernels itself; run once")
    g = torch.Generator(device="cuda").manual_seed(tiles)

    def fp8(*shape):
        return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g) & 0xBF  # finite values below 2

    def scale(*shape):
        return torch.exp2(torch.randint(-6, 3, shape, device="cuda", generator=g).float())

    def both(make):
        out = []
        for kernel in (b"r0", b"s128"):
            _lib.call("pt_gemm_select_kernel", kernel)
            out.append(make())
        assert torch.equal(*out)

    rows = torch.tensor([128, 0, 640, 1024, 1152, 0, 2688], dtype=torch.int32)  # 1, 3, 4, 5 and 11 row tiles
    G_, M, N, K = len(rows), int(rows.sum()), 256 * tiles - 112, 256
    offs = torch.cumsum(rows, 0).int().cuda()
    a, sa, b, sb = fp8(M, K), scale(M, K // 128), fp8(G_, N, K), scale(G_, (N + 127) // 128, K // 128)

    def m_grouped():
        o = torch.zeros((M, N), dtype=torch.bfloat16, device="cuda")
        _lib.call("pt_gemm_m_grouped_nt", _lib.ptr(a), _lib.ptr(sa), _lib.ptr(b), _lib.ptr(sb), _lib.ptr(o), _lib.dtype_code(o.dtype),
                  _lib.ptr(offs), G_, M, N, K, _lib.stream_ptr())
        return o

    both(m_grouped)
    for W in (256 * 4, 256 * 11 - 128):  # the other side of a weight gradient
        d, sd, x, sx = fp8(N, M), scale(M // 128, N), fp8(W, M), scale(M // 128, W)

        def k_grouped():
            o = torch.zeros((G_, N, W), dtype=torch.bfloat16, device="cuda")
            _lib.call("pt_gemm_k_grouped_wgrad", _lib.ptr(d), _lib.ptr(sd), _lib.ptr(x), _lib.ptr(sx), _lib.ptr(o), _lib.dtype_code(o.dtype), 0,
                      _lib.ptr(offs), G_, M, N, W, _lib.stream_ptr())
            return o

        both(k_grouped)


def test_grouped_work_lists_longer_than_the_tile_table(gemm_kernel):
    """12800 large tiles, 50 for every workgroup, so that the table is filled a second time from the scan that the
    first one was made of: the bits of the kernel that takes one small tile per workgroup.  m-grouped, then
    k-grouped with empty groups among them."""
    from pith_train_amd import _lib

    if gemm_kernel != "auto":
        pytest.skip("the test selects the kernels itself; run once")

    def both(make):
        out = []
        for kernel in (b"r0", b"s128"):
            _lib.call("pt_gemm_select_kernel", kernel)
            out.append(make())
        assert torch.equal(*out)

    def fp8(*shape, seed):
        g = torch.Generator(device="cuda").manual_seed(seed)
        return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g) & 0xBF  # finite values below 2

    def scale(*shape, seed):
        g = torch.Generator(device="cuda").manual_seed(seed)
        return torch.exp2(torch.randint(-6, 3, shape, device="cuda", generator=g).float())

    G_, N, K = 100, 32768, 128
    a, sa, b, sb = fp8(G_ * 128, K, seed=1), scale(G_ * 128, 1, seed=2), fp8(G_, N, K, seed=3), scale(G_, N // 128, 1, seed=4)
    offs = torch.arange(1, G_ + 1, dtype=torch.int32, device="cuda") * 128

    def m_grouped():
        o = torch.empty((G_ * 128, N), dtype=torch.bfloat16, device="cuda")
        _lib.call("pt_gemm_m_grouped_nt", _lib.ptr(a), _lib.ptr(sa), _lib.ptr(b), _lib.ptr(sb), _lib.ptr(o), _lib.dtype_code(o.dtype),
                  _lib.ptr(offs), G_, G_ * 128, N, K, _lib.stream_ptr())
        return o

    both(m_grouped)
    ks = torch.tensor([128, 0, 256, 128] * 32, dtype=torch.int32)
    offs_k, M, W = torch.cumsum(ks, 0).int().cuda(), int(ks.sum()), 2560
    d, sd, x, sx = fp8(W, M, seed=5), scale(M // 128, W, seed=6), fp8(W, M, seed=7), scale(M // 128, W, seed=8)

    def k_grouped():
        o = torch.empty((128, W, W), dtype=torch.bfloat16, device="cuda")
        _lib.call("pt_gemm_k_grouped_wgrad", _lib.ptr(d), _lib.ptr(sd), _lib.ptr(x), _lib.ptr(sx), _lib.ptr(o), _lib.dtype_code(o.dtype), 0,
                  _lib.ptr(offs_k), 128, M, W, W, _lib.stream_ptr())
        return o

    both(k_grouped)


@pytest.mark.parametrize("groups,big,rest,N,W,form", [
    (2, (300, 40), 0, 1024, 1280, "parts"),      # fewer tiles than workgroups; XCD parts that end inside a group
    (19, (90, 61, 33), 3, 1100, 1800, "parts"),  # ragged tile grid, counts of groups and tiles that no eighth divides
    (256, (130, 128, 90), 1, 512, 1024, "parts"),  # as many groups as the schedule holds, the last ones idle
    (120, (48,), 49, 256, 1280, "parts"),  # no tile of a whole share; fewer tiles a group than XCDs
    (70, (37, 36, 30), 4, 2816, 1300, "eighths"),  # remainders of tiles and of groups
    (53, (90, 80, 66), 14, 1024, 2048, "eighths"),  # the fewest tiles a group that eighths take: four each
    (45, (70, 80, 66), 24, 1500, 1400, "eighths"),  # 36 of them: four or five
])
def test_k_grouped_schedule_of_shorter_and_less_skewed_launches(gemm_kernel, groups, big, rest, N, W, form):
    """Parts, where every XCD deals out its own part of the list, and eighths of every group, at the ends of what the rule gives
    them.  Every tile once (accumulating), with the bits of one small tile per workgroup."""
    from pith_train_amd import _lib

    if gemm_kernel != "auto":
        pytest.skip("the test selects the kernels itself; run once")
    g = torch.Generator(device="cuda").manual_seed(groups)
    tiles = -(-N // 256) * -(-W // 256)
    blocks = torch.randint(0, rest + 1, (groups,), generator=torch.Generator().manual_seed(groups))
    for i, b in enumerate(big):
        blocks[i * (groups // len(big))] = b
    assert schedule(blocks.tolist(), tiles, min(256, groups * tiles))[0] == form
    offs, M = torch.cumsum(blocks * 128, 0).int().cuda(), int(blocks.sum()) * 128

    def fp8(*shape):
        return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g) & 0xBF  # finite values below 2

    def scale(*shape):
        return torch.exp2(torch.randint(-6, 3, shape, device="cuda", generator=g).float())

    d, sd, x, sx = fp8(N, M), scale(M // 128, N), fp8(W, M), scale(M // 128, W)
    start = torch.randn((groups, N, W), device="cuda", generator=g).bfloat16()
    for add in (0, 1):
        out = []
        for kernel in ("s128", "r0"):
            _lib.call("pt_gemm_select_kernel", kernel.encode())
            out.append(start.clone())
            _lib.call("pt_gemm_k_grouped_wgrad", _lib.ptr(d), _lib.ptr(sd), _lib.ptr(x), _lib.ptr(sx), _lib.ptr(out[-1]), _lib.dtype_code(torch.bfloat16),
                      add, _lib.ptr(offs), groups, M, N, W, _lib.stream_ptr())
        assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("groups,half,W", [(40, 640, 1800), (256, 896, 2200)])
def test_k_grouped_schedule_with_two_outputs_and_a_second_table(gemm_kernel, groups, half, W):
    """The rows of a gate and of an up projection go to two gradients, whose border lies inside a row of tiles, under the
    schedule of skewed groups; with 256 groups the workgroups that get small tiles alone take more than the 48 that
    the tile table holds.  The bits of one small tile per workgroup into one output."""
    from pith_train_amd import _lib

    if gemm_kernel != "auto":
        pytest.skip("the test selects the kernels itself; run once")
    g = torch.Generator(device="cuda").manual_seed(groups)
    N = 2 * half
    tiles = -(-N // 256) * -(-W // 256)
    blocks = torch.randint(0, 2, (groups,), generator=torch.Generator().manual_seed(groups))
    blocks[groups // 3] = 60 if groups == 256 else int(1.3 * 96 * 256 / tiles)
    form, share, _ = schedule(blocks.tolist(), tiles)
    assert form != "in order"
    assert groups != 256 or share / 4 > 52  # small tiles cost 3 or 4: a workgroup without a big one
    offs, M = torch.cumsum(blocks * 128, 0).int().cuda(), int(blocks.sum()) * 128

    def fp8(*shape):
        return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g) & 0xBF  # finite values below 2

    def scale(*shape):
        return torch.exp2(torch.randint(-6, 3, shape, device="cuda", generator=g).float())

    d, sd, x, sx = fp8(N, M), scale(M // 128, N), fp8(W, M), scale(M // 128, W)
    start = torch.randn((groups, N, W), device="cuda", generator=g).bfloat16()
    operands = _lib.ptr(d), _lib.ptr(sd), _lib.ptr(x), _lib.ptr(sx)
    for add in (0, 1):
        _lib.call("pt_gemm_select_kernel", b"s128")
        want = start.clone()
        rest = _lib.dtype_code(want.dtype), add, _lib.ptr(offs), groups, M, N, W, _lib.stream_ptr()
        _lib.call("pt_gemm_k_grouped_wgrad", *operands, _lib.ptr(want), *rest)
        _lib.call("pt_gemm_select_kernel", b"r0")
        one, gate, up = start.clone(), start[:, :half].contiguous(), start[:, half:].contiguous()
        _lib.call("pt_gemm_k_grouped_wgrad", *operands, _lib.ptr(one), *rest)
        _lib.call("pt_gemm_k_grouped_wgrad_pair", *operands, _lib.ptr(gate), _lib.ptr(up), half, *rest)
        assert torch.equal(one, want)
        assert torch.equal(gate, want[:, :half]) and torch.equal(up, want[:, half:])
