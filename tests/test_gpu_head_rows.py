"""The head's row work in single launches: the stable partition, the statistics written through it, the
loss and the scaled dX, against the same steps in tensor operations: whole numbers, copied values
and products of the same order bit for bit, the loss within the rounding of an fp32 sum."""

import pytest
import torch

from _util import DEV

pytestmark = pytest.mark.gpu

V = 1003


def _rows(N, seed, live=0.6):
    g = torch.Generator(device=DEV).manual_seed(seed)
    target = torch.randint(-3, V + 3, (N,), generator=g, device=DEV)
    cew = torch.rand(N, generator=g, device=DEV)
    cew[torch.rand(N, generator=g, device=DEV) > live] = 0.0
    ok = (target >= 0) & (target < V)
    cew[~ok] = float("nan")  # an ignored row's weight is not read as one
    return target, cew, ok & (cew != 0), g


@pytest.mark.parametrize("N", [1, 2, 63, 64, 1023, 1024, 1025, 5000, 70001])
def test_partition_and_loss(N):
    from solution.body import _hip

    for live_share in (0.0, 0.6, 1.1):
        target, cew, live, g = _rows(N, N, live_share)
        perm, inv, n_live = _hip.head_partition(target, cew, V)
        want = torch.cat((live.nonzero().squeeze(1), (~live).nonzero().squeeze(1)))
        assert torch.equal(perm.long(), want) and int(n_live) == int(live.sum())
        assert torch.equal(perm[inv.long()].long(), torch.arange(N, device=DEV))
        ce = torch.randn(N, generator=g, device=DEV)
        has = (target >= 0) & (target < V)
        terms = torch.where(has, cew.double() * ce.double(), 0.0)
        got = _hip.head_loss(target, cew, ce, V)
        assert abs(float(got) - float(terms.sum())) <= 1e-6 * (float(terms.abs().sum()) + 1e-30)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("N,width", [(1, V), (77, V), (300, 1008)])
def test_rows_through_the_partition(N, width, dtype):
    from solution.body import _hip

    target, cew, live, g = _rows(N, N + 1)
    z = (torch.randn(N, width, generator=g, device=DEV) * 4).to(dtype)
    perm, inv, n_live = _hip.head_partition(target, cew, width)
    live = (target >= 0) & (target < width) & (cew != 0)

    def outs(n, amax):
        return [torch.full((n,), 7.0, device=DEV) for _ in range(3)] + [
            torch.full((n,), 7, device=DEV, dtype=amax)]

    za = z.clone()
    lse, tl, ent, amax = outs(N, torch.int32)
    _hip.head_row_softmax(za, target, torch.where(live, cew, 0.0), lse, tl, ent, amax, True, 1024.0)
    zb = z.index_select(0, perm)
    lse2, tl2, ent2, amax2 = outs(N, torch.int64)
    ce = torch.full_like(lse, 7.0)
    half = N // 2  # two chunks, as the op walks them
    for a, b in ((0, half), (half, N)):
        _hip.head_row_softmax(zb[a:b], target, cew, lse2, tl2, ent2, amax2, True, 1024.0,
                              perm=perm[a:b], ce=ce)
    for x, y in ((lse, lse2), (tl, tl2), (ent, ent2), (amax.long(), amax2), (za, zb[inv.long()])):
        assert torch.equal(x, y)
    has = (target >= 0) & (target < width)
    assert torch.equal(ce, torch.where(has, lse - tl, 0.0))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,H", [(1, 8), (300, 72), (1000, 1536)])
def test_dx(N, H, dtype):
    from solution.body import _hip

    target, cew, live, g = _rows(N, N + H)
    perm, inv, n_live = _hip.head_partition(target, cew, V)
    prod = torch.randn(int(n_live), H, generator=g, device=DEV)
    dloss = torch.tensor(3.7, device=DEV)
    dx = torch.full((N, H), float("nan"), device=DEV, dtype=dtype)
    _hip.head_dx(prod, inv, cew, dloss, 1024.0, dx)
    want = torch.zeros(N, H, device=DEV)
    rows = perm[:int(n_live)].long()
    want[rows] = prod * (cew[rows] * (1.0 / 1024.0)).unsqueeze(1)
    assert torch.equal(dx, (want * dloss).to(dtype))


def test_odd_width_and_recorded_backward():
    """A width the dX kernel does not take, and a backward pass that is itself recorded (the
    gradient of the loss's own gradient reaches a factor in front of it)."""
    from solution.head import fused_linear_ce

    g = torch.Generator(device=DEV).manual_seed(3)
    target, cew, live, _ = _rows(50, 9)
    cew = torch.where(live, cew, 0.0)
    for H in (12, 64):
        x = torch.randn(50, H, generator=g, device=DEV, requires_grad=True)
        w = (torch.randn(V, H, generator=g, device=DEV) * 0.1).half()
        c = torch.tensor(2.0, device=DEV, requires_grad=True)
        loss, _ = fused_linear_ce(x, w, target, cew)
        (plain,) = torch.autograd.grad(loss, x, retain_graph=True)
        (dx,) = torch.autograd.grad(loss * c, x, create_graph=True)
        (dc,) = torch.autograd.grad(dx.sum(), c)
        torch.testing.assert_close(dx, 2 * plain, rtol=1e-6, atol=0)
        torch.testing.assert_close(dc, plain.sum(), rtol=1e-3, atol=1e-7)
        assert bool((plain[~live] == 0).all()) and bool((plain[live] != 0).any())


def _loss(seed, dtype=torch.float32):
    from solution.head import fused_linear_ce

    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(50, 64, generator=g, device=DEV).to(dtype).requires_grad_()
    w = (torch.randn(V, 64, generator=g, device=DEV) * 0.1).half()
    target, cew, live, _ = _rows(50, seed)
    cew = torch.where(live, cew, 0.0)
    loss, _ = fused_linear_ce(x, w, target, cew)
    return x, cew, live, loss


def test_weights_refilled_before_backward():
    """The caller's ce_weight is read by the forward only: its buffer may be refilled before the backward
    pass."""
    x, cew, _, loss = _loss(4)
    (want,) = torch.autograd.grad(loss, x, retain_graph=True)
    cew.fill_(3.0)
    (got,) = torch.autograd.grad(loss, x)
    assert torch.equal(got, want)


def test_weights_from_inference_mode():
    from solution.head import fused_linear_ce

    with torch.inference_mode():
        cew = torch.rand(20, device=DEV)
    x = torch.randn(20, 64, device=DEV, requires_grad=True)
    w, target = torch.randn(V, 64, device=DEV).half(), torch.arange(20, device=DEV)
    (got,) = torch.autograd.grad(fused_linear_ce(x, w, target, cew)[0], x)
    (want,) = torch.autograd.grad(fused_linear_ce(x, w, target, cew.clone())[0], x)
    assert torch.equal(got, want)


@pytest.mark.parametrize("dloss", [float("inf"), float("-inf"), float("nan")])
def test_gradient_of_a_loss_that_overflowed(dloss):
    """dX is the finished gradient times the loss's: a non-finite one marks every row, also those without
    a loss (0 * inf), in the kernel as in the tensor operations (odd widths, recorded passes)."""
    x, _, live, loss = _loss(6, torch.float16)
    assert bool(live.any()) and not bool(live.all())
    (got,) = torch.autograd.grad(loss, x, torch.tensor(dloss, device=DEV), retain_graph=True)
    scale = torch.tensor(dloss, device=DEV, requires_grad=True)
    (want,) = torch.autograd.grad(loss, x, scale, create_graph=True)
    torch.testing.assert_close(got, want.detach(), rtol=0, atol=0, equal_nan=True)
    assert not bool(torch.isfinite(got[~live]).any())
