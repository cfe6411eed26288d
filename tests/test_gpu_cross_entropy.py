"""GPU parity: in-place fused cross-entropy through the C-ABI vs the oracle.

The loss agrees to 1e-5 (fp32 statistics in another summation order, hardware exp2); a gradient
entry is the oracle's to one rounding step of the logits' dtype, and bit-equal wherever the
arithmetic is exact (uniform logits, ignored rows, the scaling of the backward)."""

import math

import pytest
import torch

from oracle import cross_entropy as CE

pytestmark = pytest.mark.gpu


def _case(N, V, seed, dtype, ignore_frac=0.2):
    g = torch.Generator().manual_seed(seed)
    x = (torch.randn((N, V), generator=g) * 3).to(dtype)
    y = torch.randint(0, V, (N,), generator=g)
    y[torch.rand(N, generator=g) < ignore_frac] = -100
    return x, y


def _check_grad(got, ref, dtype, least=1e-30):
    got, ref = got.float().cpu(), ref.float()
    assert got.shape == ref.shape
    if got.numel() == 0:
        return
    if dtype == torch.float32:
        torch.testing.assert_close(got, ref, rtol=2e-5, atol=1e-10)
        return
    step = 2.0**-7 if dtype == torch.bfloat16 else 2.0**-10
    assert ((got - ref).abs() <= ref.abs() * step + least).all(), "more than one rounding step apart"
    assert (got == ref).float().mean() > 0.98


@pytest.mark.parametrize("N,V,dtype", [
    (64, 4096, torch.bfloat16), (33, 151936, torch.bfloat16), (16, 50000, torch.float32), (9, 1000, torch.float16),
    (7, 1003, torch.bfloat16),   # V not a multiple of 8: rows that start inside a chunk
    (3, 5, torch.float32), (1, 201088, torch.bfloat16), (0, 128, torch.bfloat16),
])
def test_forward_backward(N, V, dtype):
    from pith_train_amd.operators.cross_entropy import cross_entropy

    x, y = _case(N, V, N + V, dtype)
    o_loss, o_grad, _, _ = CE.cross_entropy_fwd(x, y)
    leaf = x.cuda().requires_grad_(True)
    buf = leaf.clone()  # the operator overwrites its input: hand it a non-leaf
    loss = cross_entropy(buf, y.cuda())
    assert loss.dtype == torch.float32 and loss.shape == ()
    torch.testing.assert_close(loss.cpu(), o_loss, rtol=1e-5, atol=1e-6)
    _check_grad(buf.detach(), o_grad, dtype)  # the forward already left the gradient in place
    stored = buf.detach().clone()
    (loss * 0.3).backward()
    assert torch.equal(leaf.grad, stored * torch.tensor(0.3).to(dtype))  # one multiplication: no freedom
    if N:
        # a unit incoming gradient leaves the stored gradient as it is
        leaf2 = x.cuda().requires_grad_(True)
        buf2 = leaf2.clone()
        cross_entropy(buf2, y.cuda()).backward()
        assert torch.equal(leaf2.grad, stored)


def test_exact_cases():
    from pith_train_amd.operators.cross_entropy import cross_entropy

    N, V = 4, 512
    x = torch.full((N, V), 1.25, dtype=torch.bfloat16).cuda()
    y = torch.tensor([0, 5, 511, 7])
    loss = cross_entropy(x, y.cuda())
    assert abs(float(loss) - math.log(V)) < 1e-6
    want = torch.full((N, V), 2.0**-11).bfloat16()
    want[torch.arange(N), y] = torch.tensor(2.0**-11 - 0.25).bfloat16()
    assert torch.equal(x.cpu(), want)
    # two roundings at the target: the stored softmax term is corrected afterwards
    x = torch.tensor([[0.0, math.log(3.0)] + [-1e4] * 6]).bfloat16().cuda()
    cross_entropy(x, torch.tensor([1]).cuda())
    assert float(x[0, 1]) == float((torch.tensor(0.75).bfloat16().float() - 1.0).bfloat16())


def test_ignore_rules_and_masked_vocabulary():
    from pith_train_amd.operators.cross_entropy import cross_entropy

    x, y = _case(9, 304, 1, torch.bfloat16, ignore_frac=0.0)
    y[[2, 5]] = -100
    buf = x.cuda()
    loss = cross_entropy(buf, y.cuda())
    o_loss, o_grad, _, _ = CE.cross_entropy_fwd(x, y)
    torch.testing.assert_close(loss.cpu(), o_loss, rtol=1e-5, atol=1e-6)
    assert buf[[2, 5]].abs().max() == 0
    buf = x.cuda()
    loss = cross_entropy(buf, torch.full((9,), -100).cuda())  # nothing counts: n clamps to 1
    assert float(loss) == 0 and buf.abs().max() == 0
    buf = x.cuda()
    loss = cross_entropy(buf, torch.full((9,), 7).cuda(), ignore_index=7)
    assert float(loss) == 0 and buf.abs().max() == 0
    # a vocabulary whose tail is masked with -inf: zero probability there, finite loss
    xm = x.clone()
    xm[:, 200:] = float("-inf")
    ym = y.clamp(min=0) % 200
    o_loss, o_grad, _, _ = CE.cross_entropy_fwd(xm, ym)
    buf = xm.cuda()
    loss = cross_entropy(buf, ym.cuda())
    torch.testing.assert_close(loss.cpu(), o_loss, rtol=1e-5, atol=1e-6)
    assert buf[:, 200:].abs().max() == 0 and torch.isfinite(buf).all()


def test_full_size_rows_sum_to_zero_and_loss_matches_torch():
    """2048 rows of a 151 936-entry vocabulary: the loss equals torch's cross_entropy on the same
    device, every gradient row of a counted token sums to zero (softmax minus one-hot) within the
    bf16 rounding of its entries, and two runs give the same bits."""
    import torch.nn.functional as F

    from pith_train_amd.operators.cross_entropy import cross_entropy

    N, V = 2048, 151936
    g = torch.Generator(device="cuda").manual_seed(5)
    x = (torch.randn((N, V), device="cuda", generator=g) * 2).bfloat16()
    y = torch.randint(0, V, (N,), device="cuda", generator=g)
    y[::7] = -100
    ref = F.cross_entropy(x.float(), y, ignore_index=-100)
    a, b = x.clone(), x.clone()
    la, lb = cross_entropy(a, y), cross_entropy(b, y)
    assert torch.equal(la, lb) and torch.equal(a, b)
    torch.testing.assert_close(la, ref, rtol=1e-5, atol=1e-6)
    n = int((y != -100).sum())
    sums = a.float().sum(-1) * n
    assert sums[y == -100].abs().max() == 0
    assert sums[y != -100].abs().max() < 2e-2


@pytest.mark.parametrize("N,V,dtype", [(256, 264, torch.bfloat16), (257, 8, torch.bfloat16), (515, 125000, torch.float16), (600, 122880, torch.bfloat16)])
def test_more_rows_than_workgroups(N, V, dtype):
    """A workgroup that walks several rows gives each of them what a workgroup of its own gives: rows within
    the registers, exactly as long as they hold, and past them; ignored rows in every position."""
    from pith_train_amd.operators.cross_entropy import cross_entropy

    g = torch.Generator(device="cuda").manual_seed(N)
    x = (torch.randn((N, V), device="cuda", generator=g) * 2).to(dtype)
    y = torch.randint(0, V, (N,), device="cuda", generator=g)
    y[::5] = -100
    whole = x.clone()
    loss = cross_entropy(whole, y)
    total = torch.zeros((), dtype=torch.float64, device="cuda")
    n = int((y != -100).sum())
    for r0 in range(0, N, 128):
        part, yp = x[r0 : r0 + 128].clone(), y[r0 : r0 + 128]
        np_ = max(1, int((yp != -100).sum()))
        total += cross_entropy(part, yp).double() * np_
        a, b = whole[r0 : r0 + 128].float() * n, part.float() * np_  # both rounded after the division by their own n
        step = 2.0 ** (-6 if dtype == torch.bfloat16 else -9)
        at_target = torch.zeros_like(b)  # there the softmax term was rounded before 1 was taken off
        at_target[torch.arange(len(yp), device="cuda"), yp.clamp(min=0)] = step
        assert ((a - b).abs() <= step * b.abs() + at_target + (2.0 ** -20 if dtype == torch.float16 else 1e-20) * n).all()
    torch.testing.assert_close(loss.double(), total / n, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("N,V,start", [
    (19, 1, 0), (19, 3, 1), (19, 9, 5),  # rows that are edges alone, or hold one chunk or none
    (600, 1003, 0),      # more rows than compute units: a row's neighbour starts elsewhere in a chunk
    (260, 50257, 3),
    (3, 32767, 1), (3, 32776, 0), (3, 16384, 3),  # the longest of the short rows and the next, of 16 and of 32 bits
    (3, 61441, 1), (2, 122888, 7),  # as long as the registers hold, and a chunk more or less by where a row starts
    (2, 204665, 0), (2, 102337, 2),  # as long as registers and LDS hold, of 16 and of 32 bits; past it the row is read twice
    (2, 300007, 6),
])
def test_rows_that_start_anywhere(N, V, start, dtype):
    """Rows of a length that is no multiple of a chunk, in a buffer that starts inside one: targets among the first and the
    last elements of a row, and nothing written outside of the rows."""
    from pith_train_amd.operators.cross_entropy import cross_entropy

    x, y = _case(N, V, N + V, dtype)
    y[::3] = torch.arange(len(y[::3])) % min(V, 9)
    y[1::3] = V - 1 - torch.arange(len(y[1::3])) % min(V, 9)
    y[-1] = -100
    o_loss, o_grad, _, _ = CE.cross_entropy_fwd(x, y)
    flat = torch.full((start + N * V + 16,), 7.0, dtype=dtype, device="cuda")
    buf = flat[start : start + N * V].view(N, V)
    buf.copy_(x)
    buf.requires_grad_(True)
    loss = cross_entropy(buf.view(N, V), y.cuda())
    torch.testing.assert_close(loss.detach().cpu(), o_loss, rtol=1e-5, atol=1e-6)
    stored = buf.detach().clone()
    # (rows of 300 007: float16 gradients below 2^-14 are 2^-24 apart, one step of which is more than 2^-10 of them)
    _check_grad(stored, o_grad, dtype, 2.0**-24 if dtype == torch.float16 else 1e-30)
    (grad,) = torch.autograd.grad(loss * 0.3, buf)
    assert torch.equal(grad, stored * torch.tensor(0.3).to(dtype))
    assert (flat[:start] == 7).all() and (flat[start + N * V :] == 7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("V", [3, 9, 304, 1003, 4096, 32776, 102337, 204665, 300007])
def test_a_nan_among_masked_logits_is_seen(V, dtype):
    """A logit that is not a number makes the loss and its row's gradient so, wherever it stands: at the ends of a row, which
    single threads read, and between -inf logits, with which it is all that a thread sees."""
    from pith_train_amd.operators.cross_entropy import cross_entropy

    places = sorted({p for p in (0, 1, 5, V // 2, V // 2 + 3, V - 2, V - 1) if 0 <= p < V})
    x, _ = _case(len(places) + 1, V, V, dtype)
    for row, p in enumerate(places):
        x[row, max(p - 3, 0) : p + 4] = -math.inf
        x[row, p] = math.nan
    y = torch.full((len(x),), V // 3)
    for row in range(len(places)):
        buf = x[[row, -1]].cuda()
        loss = cross_entropy(buf, y[:2].cuda())
        assert math.isnan(float(loss)), places[row]
        assert buf[0].isnan().all() and buf[1].isfinite().all()
