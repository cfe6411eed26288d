"""The small-problem GEMM kernel (64- and 128-row tiles) against the persistent kernels: same MFMAs in
the same order, so the same bits, at the edges of its tiles and of its reduction stages."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _fp8(g, *shape):
    return (torch.randn(shape, generator=g) * 60).to(torch.float8_e4m3fn).cuda()


def _scale(g, *shape):
    return torch.exp2(torch.randint(-8, 2, shape, generator=g).float()).cuda()


def _cdiv(a, b):
    return -(-a // b)


def _same_bits(run, out, reference):
    from pith_train_amd import _lib

    results = {}
    for name in (reference, "s64", "s128"):
        _lib.call("pt_gemm_select_kernel", name.encode())
        try:
            out.fill_(0.5)
            run()
            torch.cuda.synchronize()
            results[name] = out.clone()
        finally:
            _lib.call("pt_gemm_select_kernel", None)
    for name in ("s64", "s128"):
        assert torch.equal(results[name], results[reference]), f"{name} differs from {reference}"


@pytest.mark.parametrize("m,n,k", [(1, 8, 16), (64, 128, 128), (65, 129, 144), (1001, 512, 2048), (130, 1003, 656), (128, 264, 5 * 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_dense(m, n, k, dtype):
    from pith_train_amd import _lib

    g = torch.Generator().manual_seed(m + n + k)
    a, sa, b, sb = _fp8(g, m, k), _scale(g, m, _cdiv(k, 128)), _fp8(g, n, k), _scale(g, _cdiv(n, 128), _cdiv(k, 128))
    out = torch.empty((m, n), device="cuda", dtype=dtype)
    _same_bits(lambda: _lib.call("pt_gemm_nt_dense", a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), out.data_ptr(),
                                 _lib.dtype_code(dtype), m, n, k, _lib.stream_ptr()), out, "q0")


@pytest.mark.parametrize("rows,n,k", [([128, 0, 384, 128], 264, 400), ([256] * 3, 128, 128), ([128] * 70, 72, 1040)])
@pytest.mark.parametrize("form", ["nt", "nn", "nn_scatter", "wgrad", "wgrad_add"])
def test_grouped(rows, n, k, form):
    from pith_train_amd.operators.grouped_linear import k_grouped_fp8_wgrad, m_grouped_fp8_gemm_nn, m_grouped_fp8_gemm_nt

    g = torch.Generator().manual_seed(n + k)
    if form != "nt":
        n = _cdiv(n, 16) * 16
    G, M = len(rows), sum(rows)
    offs = torch.tensor(rows).cumsum(0).to(torch.int32).cuda()
    if form.startswith("wgrad"):
        dy, dys, x, xs = _fp8(g, n, M), _scale(g, M // 128, n), _fp8(g, k, M), _scale(g, M // 128, k)
        out = torch.empty((G, n, k), device="cuda", dtype=torch.bfloat16)
        _same_bits(lambda: k_grouped_fp8_wgrad((dy, dys), (x, xs), out, offs, form == "wgrad_add"), out, "r0")
        return
    cap = M + 256  # a buffer sized for more rows than the routing produced
    a, sa = _fp8(g, cap, k), _scale(g, cap, _cdiv(k, 128))
    out = torch.empty((cap, n), device="cuda", dtype=torch.bfloat16)
    if form == "nt":
        b, sb = _fp8(g, G, n, k), _scale(g, G, _cdiv(n, 128), _cdiv(k, 128))
        _same_bits(lambda: m_grouped_fp8_gemm_nt((a, sa), (b, sb), out, offs), out, "r0")
        return
    b, sb = _fp8(g, G, k, n), _scale(g, G, _cdiv(k, 128), _cdiv(n, 128))
    index = None
    if form == "nn_scatter":
        index = torch.randperm(cap, generator=g).to(torch.int32)
        index[::7] = -1
        index = index.cuda()
    _same_bits(lambda: m_grouped_fp8_gemm_nn((a, sa), (b, sb), out, offs, index), out, "r0")


@pytest.mark.parametrize("m,n,k", [(1001, 4096, 1792), (4090, 1000, 2064), (129, 8, 4096), (1, 16, 1808)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_one_deep_workgroup_per_unit(m, n, k, dtype):
    """The form of the 128-row tiles with eight waves and four stages, forced and where the library picks it: the bits of the
    large tiles', with ragged rows, columns and reductions, more stages than blocks left over at the end, one row."""
    from pith_train_amd import _lib

    g = torch.Generator().manual_seed(m)
    a, sa, b, sb = _fp8(g, m, k), _scale(g, m, _cdiv(k, 128)), _fp8(g, n, k), _scale(g, _cdiv(n, 128), _cdiv(k, 128))
    results = []
    try:
        for kernel in (b"r0", b"s128d", b"auto"):
            _lib.call("pt_gemm_select_kernel", kernel)
            results.append(torch.full((m, n), 0.5, device="cuda", dtype=dtype))
            _lib.call("pt_gemm_nt_dense", a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), results[-1].data_ptr(), _lib.dtype_code(dtype),
                      m, n, k, _lib.stream_ptr())
    finally:
        _lib.call("pt_gemm_select_kernel", None)
    assert all(torch.equal(r, results[0]) for r in results)


@pytest.mark.parametrize("first,second", [((4000, 512, 4096), (4096, 512, 4000)), ((700, 2048, 2048), (2048, 2048, 704)), ((901, 2048, 4096), (4096, 2048, 912)),
                                          ((300, 4096, 2064), (2056, 4096, 304))])
def test_two_products_of_deep_tiles(first, second):
    """Pairs of long and short reductions at the rule's two sides: the bits of two launches."""
    test_two_products_in_one_launch(first, second, torch.bfloat16)


@pytest.mark.parametrize("first,second", [((1, 16, 16), (70, 24, 144)), ((1001, 2048, 512), (512, 2048, 1008)), ((640, 264, 400), (129, 1000, 272)),
                                          ((2048, 2048, 256), (2048, 2048, 128)), ((4096, 2048, 128), (128, 128, 128))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_two_products_in_one_launch(first, second, dtype):
    """Pairs that share a launch of 64- or 128-row tiles, and pairs that are too large for one."""
    import struct

    from pith_train_amd import _lib

    g = torch.Generator().manual_seed(first[0])
    block, got, want, keep = b"", [], [], []
    for m, n, k in (first, second):
        a, sa, b, sb = _fp8(g, m, k), _scale(g, m, _cdiv(k, 128)), _fp8(g, n, k), _scale(g, _cdiv(n, 128), _cdiv(k, 128))
        keep.append((a, sa, b, sb))
        got.append(torch.full((m, n), 0.5, device="cuda", dtype=dtype))
        want.append(torch.empty((m, n), device="cuda", dtype=dtype))
        _lib.call("pt_gemm_nt_dense", a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), want[-1].data_ptr(), _lib.dtype_code(dtype),
                  m, n, k, _lib.stream_ptr())
        block += struct.pack("=10q", a.data_ptr(), k, sa.data_ptr(), b.data_ptr(), k, sb.data_ptr(), got[-1].data_ptr(), m, n, k)
    _lib.call("pt_gemm_nt_dense_pair", block, _lib.dtype_code(dtype), _lib.stream_ptr())
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("rows,n,k", [([64, 0, 192, 128, 64], 264, 400), ([64] * 70, 72, 1040), ([0, 64], 8, 16)])
@pytest.mark.parametrize("scatter,bias", [(False, False), (True, False), (False, True), (True, True)])
def test_groups_of_a_few_rows(rows, n, k, scatter, bias):
    """Group ends at odd multiples of 64, against one dense product per group."""
    from pith_train_amd import _lib

    g = torch.Generator().manual_seed(n + k)
    G, M, cap = len(rows), sum(rows), sum(rows) + 128
    offs = torch.tensor(rows).cumsum(0).to(torch.int32).cuda()
    a, sa = _fp8(g, cap, k), _scale(g, cap, _cdiv(k, 128))
    b, sb = _fp8(g, G, n, k), _scale(g, G, _cdiv(n, 128), _cdiv(k, 128))
    bias_rows = torch.randn((G, n), generator=g).bfloat16().cuda() if bias else None
    index = torch.randperm(cap, generator=g).to(torch.int32).cuda() if scatter else None
    out = torch.zeros((cap, n), device="cuda", dtype=torch.bfloat16)
    _lib.call("pt_gemm_m_grouped_nt_few_rows", a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), out.data_ptr(), _lib.PT_BF16,
              offs.data_ptr(), G, cap, n, k, _lib.ptr(index), cap, _lib.ptr(bias_rows), _lib.stream_ptr())
    want, row = torch.zeros_like(out), 0
    for q, r in enumerate(rows):
        if r:
            y = torch.empty((r, n), device="cuda", dtype=torch.bfloat16)
            _lib.call("pt_gemm_nt_dense", a[row:].data_ptr(), sa[row:].data_ptr(), b[q].data_ptr(), sb[q].data_ptr(), y.data_ptr(),
                      _lib.PT_BF16, r, n, k, _lib.stream_ptr())
            y = y + bias_rows[q] if bias else y
            if scatter:
                want[index[row : row + r].long()] = y
            else:
                want[row : row + r] = y
        row += r
    assert row == M and torch.equal(out, want)


@pytest.mark.parametrize("G,n,k", [(66, 1000, 2048), (70, 15000, 128), (64, 1024, 2048), (9, 7304, 2048)])
@pytest.mark.parametrize("scatter,bias", [(False, False), (True, True)])
def test_groups_of_a_few_rows_whose_weights_are_streamed(G, n, k, scatter, bias):
    """Weights of 128 MiB and a little more, the least that is read past the memory-side cache: a last column tile that is
    not full (8 wide the last time), a reduction of one block, exactly 128 MiB."""
    from pith_train_amd import _lib

    assert 2**27 <= G * n * k < 2**27 * 1.01 and k % 128 == 0
    g = torch.Generator(device="cuda").manual_seed(n + k)

    def fp8(*shape):
        return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g) & 0xBF  # finite values below 2

    def scale(*shape):
        return torch.exp2(torch.randint(-8, 2, shape, device="cuda", generator=g).float())

    rows = torch.tensor([64, 0, 192, 128, 64, 64, 0], dtype=torch.int32).repeat(G)[:G]
    offs, M, cap = rows.cumsum(0).int().cuda(), int(rows.sum()), int(rows.sum()) + 128
    a, sa, b, sb = fp8(cap, k), scale(cap, k // 128), fp8(G, n, k), scale(G, _cdiv(n, 128), k // 128)
    bias_rows = torch.randn((G, n), device="cuda", generator=g).bfloat16() if bias else None
    index = torch.randperm(cap, device="cuda", generator=g).int() if scatter else None
    out = torch.zeros((cap, n), device="cuda", dtype=torch.bfloat16)
    args = [_lib.PT_BF16, offs.data_ptr(), G, cap, n, k, _lib.ptr(index), cap, _lib.ptr(bias_rows), _lib.stream_ptr()]
    _lib.call("pt_gemm_m_grouped_nt_few_rows", a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), out.data_ptr(), *args)
    want, row = torch.zeros_like(out), 0
    for q, r in enumerate(rows.tolist()):
        if r:
            y = torch.empty((r, n), device="cuda", dtype=torch.bfloat16)
            _lib.call("pt_gemm_nt_dense", a[row:].data_ptr(), sa[row:].data_ptr(), b[q].data_ptr(), sb[q].data_ptr(), y.data_ptr(),
                      _lib.PT_BF16, r, n, k, _lib.stream_ptr())
            y = y + bias_rows[q] if bias else y
            if scatter:
                want[index[row : row + r].long()] = y
            else:
                want[row : row + r] = y
        row += r
    assert row == M and torch.equal(out, want)


@pytest.mark.parametrize("clamp", [None, (1.702, 7.0)])
def test_padding_of_groups_of_a_few_rows_is_left_out(clamp):
    """Groups of 64 whose rows go back to their places: nothing is read or written for padding, eight rows at a time.  The
    bits of the form that writes every grouped row, for counts around the eights, rows left out inside a group and a whole
    tile of them; what the buffers held before does not matter."""
    from pith_train_amd.operators.fused_experts import forward_only

    counts = [1, 0, 7, 8, 9, 31, 33, 63, 64, 65, 130]
    G, K, half, H = len(counts), 400, 272, 264
    g = torch.Generator().manual_seed(3)
    ends = torch.tensor([_cdiv(c, 64) * 64 for c in counts]).cumsum(0)
    M = _cdiv(int(ends[-1]), 128) * 128 + 128  # rows behind the last group
    row_map, n = torch.full((M,), -1, dtype=torch.int32), 0
    for q, c in enumerate(counts):
        first = int(ends[q - 1]) if q else 0
        row_map[first : first + c] = torch.arange(n, n + c)
        n += c
    row_map[int(ends[5]) + 3] = -1                              # a hole
    row_map[int(ends[9]) : int(ends[9]) + 64] = -1              # a tile of the last group
    src = torch.randperm(n, generator=g).int()
    row_map = torch.where(row_map >= 0, src[row_map.clamp_min(0).long()], row_map).cuda()
    x = torch.randn((n, K), generator=g).bfloat16().cuda()
    q_gu = _fp8(g, G, 2 * half, K), _scale(g, G, _cdiv(2 * half, 128), _cdiv(K, 128))
    q_dn = _fp8(g, G, H, half), _scale(g, G, _cdiv(H, 128), _cdiv(half, 128))
    down = torch.empty((G, H, half), dtype=torch.bfloat16, device="cuda")
    biases = tuple(torch.randn((G, w), generator=g).bfloat16().cuda() for w in (2 * half, H)) if clamp else (None, None)

    def run(scatter):
        dirt = [torch.full((8 << 20,), 0xFF, dtype=torch.uint8, device="cuda") for _ in range(4)]  # buffers of not-a-numbers
        del dirt
        return forward_only(x, down, ends.int().cuda(), q_gu, q_dn, row_map, scatter=scatter, clamp=clamp, biases=biases, few_rows=True)

    grouped, placed = run(False), run(True)
    rows = (row_map >= 0).nonzero().squeeze(1)
    assert placed.shape == (n, H) and torch.equal(placed[row_map[rows].long()], grouped[rows])
    assert placed[row_map[rows].long()].float().abs().sum() > 0


@pytest.mark.parametrize("form", ["nt", "nn", "scatter", "nn scatter"])
def test_weights_past_the_memory_side_cache_in_tiles_of_128_rows(form):
    """Weights of 128 MiB and more of whole lines are loaded past that cache: the bits of the large tiles' kernel, for one,
    several and no tile of rows a group."""
    from pith_train_amd import _lib
    from pith_train_amd.operators.grouped_linear import m_grouped_fp8_gemm_nn, m_grouped_fp8_gemm_nt

    g = torch.Generator().manual_seed(5)
    G, N, K = 68, 1024, 2048
    rows = torch.tensor([128, 0, 384] + [128] * (G - 4) + [256])
    offs, M = rows.cumsum(0).int().cuda(), int(rows.sum())
    a = _fp8(g, M, K), _scale(g, M, K // 128)
    nn = "nn" in form
    gemm = m_grouped_fp8_gemm_nn if nn else m_grouped_fp8_gemm_nt
    one = _fp8(g, 1, K, N) if nn else _fp8(g, 1, N, K)
    b = one.view(torch.uint8).repeat(G, 1, 1)
    b[G // 2] = b[G // 2].flip(0)
    b = b.view(one.dtype), _scale(g, G, K // 128, N // 128) if nn else _scale(g, G, N // 128, K // 128)
    assert b[0].numel() >= 128 << 20
    index = (torch.randperm(M, generator=g).int().cuda(),) if "scatter" in form else ()
    out = []
    for kernel in (b"s128", b"r0"):
        _lib.call("pt_gemm_select_kernel", kernel)
        out.append(torch.zeros((M, N), device="cuda", dtype=torch.bfloat16))
        gemm(a, b, out[-1], offs, *index)
    _lib.call("pt_gemm_select_kernel", b"auto")
    assert out[0].float().abs().sum() > 0 and torch.equal(*out)
