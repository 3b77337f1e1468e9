"""The fused LoRA products (esep_lora_down / esep_lora_up / esep_lora_grads) at the edges of their
tiles (16-row, 32-row and 64-column steps, 256-column blocks, 16-rank tiles, the chunk split),
against float64 products of the same 16-bit operands with the oracle's mask.

Bounds, with u the unit roundoff of the stored type (2^-11 fp16, 2^-8 bf16) and S the sum of the
products' magnitudes: a 16-bit result rounds once (u |want|), a dropped input is rounded before
its product (u S), and fp32 sums of at most 2^14 terms stay within 1e-5 S; 2^-24 covers fp16's
subnormal spacing."""

import numpy as np
import pytest
import torch

from _util import DEV, gen
from oracle import lora_ref as ref

pytestmark = pytest.mark.gpu

U = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


@pytest.fixture
def kernels(monkeypatch):
    """Every product on the fused kernels, also where the library is the faster one."""
    from solution.body import lora as L

    for name in ("_down_pays", "_dxa_pays", "_down_grads_pay", "_up_grads_pay", "_base_pays"):
        monkeypatch.setattr(L, name, lambda *a: True)


KEY = 0x1357_9BDF_2468_ACE

# (T, in, out, rank): one row; a ragged 16-row tile with narrow sides; ranks between tiles; the
# 64-column and 256-column edges on both sides; two chunks; several rows tiles per block
SHAPES = [(1, 8, 8, 8), (17, 72, 264, 16), (33, 200, 72, 24), (64, 520, 256, 40),
          (130, 1536, 256, 16), (1000, 1032, 1536, 64), (8200, 64, 136, 32), (16500, 128, 64, 64)]


def _close(got, want, bound, what):
    err = (got.double() - want).abs()
    assert torch.isfinite(got).all(), what
    assert bool((err <= bound + 2.0 ** -24).all()), (what, float((err - bound).max()))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("p", [0.0, 0.1])
@pytest.mark.parametrize("T,K,N,r", SHAPES)
def test_fused_products(T, K, N, r, p, dtype, kernels):
    from solution.body import lora as L

    g, u, s = gen(T + K + r), U[dtype], 2.0

    def rnd(*shape):
        return torch.randn(*shape, generator=g).to(dtype).to(DEV)

    x, a, b, base = rnd(T, K), rnd(r, K), rnd(N, r), rnd(T, N)
    wide = rnd(T, N + 16)
    dterm = wide[:, 8:8 + N]  # a column block of a wider gradient
    assert L._fused(r, x, a) and L._up_bwd_fused(dterm, rnd(T, r), b)
    key = torch.tensor([KEY], device=DEV)
    keep = torch.ones(T, K, device=DEV, dtype=torch.float64)
    if p > 0:
        m = ref.dropout_mask(KEY, T * K, float(np.float32(p)))
        keep = torch.from_numpy(m.reshape(T, K)).to(DEV).double() / (1 - p)
    xd, ux = x.double() * keep, u if p > 0 else 0.0
    A, B, D = a.double(), b.double(), dterm.double()

    xa = L.lora_down_fwd(x, a, key, p)
    want, S = xd @ A.T, xd.abs() @ A.abs().T
    _close(xa, want, u * want.abs() + (ux + 1e-5) * S, "xa")
    X = xa.double()

    term = L.lora_delta(xa, b, s)
    want, S = s * X @ B.T, s * X.abs() @ B.abs().T
    _close(term, want, u * want.abs() + 1e-5 * S, "term")
    out = L.LoRAFunction.apply(x, base.clone(), a, b, 0.0, s)
    xa0 = (L.lora_down_fwd(x, a, key, 0.0)).double()
    want = base.double() + s * xa0 @ B.T
    _close(out, want, u * want.abs() + 1e-5 * (s * xa0.abs() @ B.abs().T + base.double().abs()),
           "base + term")

    dxa, db = L.lora_up_bwd(dterm, xa, b, s)
    want, S = s * D @ B, s * D.abs() @ B.abs()
    _close(dxa, want, u * want.abs() + 1e-5 * S, "dxa")
    _close(db, s * D.T @ X, 1e-5 * (s * D.abs().T @ X.abs()), "dB")
    assert torch.equal(db, L.lora_up_bwd(dterm, xa, b, s)[1])

    dx, da = L.lora_down_bwd(x, a, dxa, key, p)
    G = dxa.double()
    want, S = (G @ A) * keep, (G.abs() @ A.abs()) * keep
    _close(dx, want, u * want.abs() + 1e-5 * S, "dx")
    assert not bool(dx[keep == 0].any())
    _close(da, G.T @ xd, (ux + 1e-5) * (G.abs().T @ xd.abs()), "dA")
    acc = rnd(T, K)
    dx2, da2 = L.lora_down_bwd(x, a, dxa, key, p, dx_accum=acc.clone())
    _close(dx2, acc.double() + want, u * (acc.double() + want).abs() + 1e-5 * (S + 1), "dx +=")
    none, da3 = L.lora_down_bwd(x, a, dxa, key, p, need_dx=False)
    assert none is None and torch.equal(da, da2) and torch.equal(da, da3)


def test_other_ranks_and_layouts_keep_their_path():
    """What the fused products do not take runs on the library products: ranks that are no
    multiple of 8 or above 64, odd widths, unaligned rows."""
    from solution.body import lora as L

    x = torch.randn(40, 64, device=DEV).half()
    assert not L._fused(12, x) and not L._fused(72, x) and not L._fused(16, x[:, :63])
    assert not L._fused(16, x[:, 1:57]) and not L._fused(16, x.t()) and not L._fused(16, x.float())
    for r, K in ((12, 64), (72, 64), (16, 63)):
        a, b = torch.randn(r, K, device=DEV) * 0.1, torch.randn(24, r, device=DEV) * 0.1
        xi = x[:, :K].clone().requires_grad_()
        ai, bi = a.clone().requires_grad_(), b.clone().requires_grad_()
        term = L.LoRADeltaFunction.apply(xi, ai, bi, 0.0, 2.0)
        grads = torch.autograd.grad(term, (xi, ai, bi), torch.ones_like(term))
        xr, ar, br = (t.detach().double().requires_grad_() for t in (xi, a, b))
        want = 2.0 * (xr @ ar.T) @ br.T
        wants = torch.autograd.grad(want, (xr, ar, br), torch.ones_like(want))
        for got, w in zip((term, *grads), (want, *wants)):
            # a chain of three fp16 roundings
            assert (got.double() - w).abs().max() <= 4 * 2.0 ** -11 * w.abs().max()


@pytest.mark.parametrize("p", [0.0, 0.1])
@pytest.mark.parametrize("T,K,N,r", [(200, 3584, 256, 64), (64, 8960, 64, 32), (2000, 256, 8960, 16),
                                     (6000, 1536, 64, 16)])
def test_routes_agree(T, K, N, r, p, monkeypatch):
    """Where a product goes changes its rounding alone: the whole term, forward and backward, on the
    kernels, on the library and as the rules say. Results of a chain of at most four fp16 roundings."""
    from solution.body import lora as L

    g = gen(T + K)
    x = torch.randn(T, K, generator=g).half().to(DEV).requires_grad_()
    a = (torch.randn(r, K, generator=g) * 0.05).to(DEV).requires_grad_()
    b = (torch.randn(N, r, generator=g) * 0.05).to(DEV).requires_grad_()
    base, d = (torch.randn(T, N, generator=g).half().to(DEV) for _ in range(2))
    monkeypatch.setattr(L, "new_dropout_key", lambda device: torch.tensor([KEY], device=device))
    names = ("_down_pays", "_dxa_pays", "_down_grads_pay", "_up_grads_pay", "_base_pays")
    outs = []
    for route in (True, False, None):
        with monkeypatch.context() as m:
            for name in names if route is not None else ():
                m.setattr(L, name, lambda *args, route=route: route)
            out = L.LoRAFunction.apply(x, base.clone(), a, b, p, 2.0)
            outs.append((out, *torch.autograd.grad(out, (x, a, b), d)))
    for one in outs[1:]:
        for got, want in zip(one, outs[0]):
            assert (got - want).float().abs().max() <= 4 * 2.0 ** -11 * want.float().abs().max()
