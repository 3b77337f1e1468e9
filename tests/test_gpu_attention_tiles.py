"""Varlen attention at the edges of its tiles for both head dims (32-query and 32-key steps, the 64-key
tiles of D = 64, 128-query and 128-key blocks), split and unsplit query heads, dense and strided
rows, against float64.

Bounds, with u the unit roundoff of the type (2^-11 fp16, 2^-8 bf16): a probability and a dS enter
their products rounded (u each), results round once, and delta = rowsum(dO o) is formed from the
rounded o (u sum |dO| |o|); a factor 1.05 covers fp32 sums, exponentials and second order."""

import pytest
import torch

from _util import DEV

pytestmark = pytest.mark.gpu

U = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _reference(q, k, v, do, lens, u):
    """float64 (o, dq, dk, dv) and the elementwise error bounds."""
    q, k, v, do = (t.double() for t in (q, k, v, do))
    hq, hk, d = q.shape[1], k.shape[1], q.shape[2]
    scale, t0 = d ** -0.5, 0
    out = [torch.zeros_like(x) for x in (q, q, k, v)]
    err = [torch.zeros_like(x) for x in (q, q, k, v)]
    for n in lens:
        r = slice(t0, t0 + n)
        mask = torch.ones(n, n, device=q.device, dtype=torch.bool).tril()
        for h in range(hq):
            g = h // (hq // hk)
            qs, ks, vs, ds = q[r, h], k[r, g], v[r, g], do[r, h]
            p = torch.softmax((qs @ ks.T * scale).masked_fill(~mask, float("-inf")), -1)
            o, dp = p @ vs, ds @ vs.T
            dz = p * (dp - (dp * p).sum(-1, keepdim=True))
            eo = u * (p @ vs.abs()) + u * o.abs()
            # dS's own rounding, and delta from the rounded o (error of o, then of the dot)
            edz = u * dz.abs() + p * ((ds.abs() * eo).sum(-1, keepdim=True))
            for i, (val, e) in enumerate(((o, eo), (scale * dz @ ks, scale * edz @ ks.abs()))):
                out[i][r, h], err[i][r, h] = val, e
            out[2][r, g] += scale * dz.T @ qs
            err[2][r, g] += scale * edz.T @ qs.abs()
            out[3][r, g] += p.T @ ds
            err[3][r, g] += u * p.T @ ds.abs()
        t0 += n
    return out, [e + (0 if i == 0 else u) * o.abs() for i, (o, e) in enumerate(zip(out, err))]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("hq,hk", [(7, 1), (4, 4)])
@pytest.mark.parametrize("lens", [[1], [31, 32, 33], [63, 0, 64, 65], [127, 128, 129, 1],
                                  [300, 97, 512, 2]], ids=lambda v: "-".join(map(str, v)))
def test_tile_edges(lens, hq, hk, D, dtype):
    from solution.body.attention import cu_seqlens_from_lengths, varlen_attention

    T, g = sum(lens), torch.Generator(device=DEV).manual_seed(sum(lens) + D)
    wide = torch.randn(T, hq + 2 * hk, D, generator=g, device=DEV).to(dtype)
    q, k, v = (t.detach().requires_grad_() for t in wide.split([hq, hk, hk], 1))  # strided rows
    do = torch.randn(T, hq, D, generator=g, device=DEV).to(dtype)
    o = varlen_attention(q, k, v, cu_seqlens_from_lengths(lens, DEV), max(lens))
    got = (o, *torch.autograd.grad(o, (q, k, v), do))
    want, bound = _reference(q, k, v, do, lens, U[dtype])
    for name, a, b, e in zip(("o", "dq", "dk", "dv"), got, want, bound):
        off = (a.double() - b).abs() - (1.05 * e + 2.0 ** -22)
        assert bool((off <= 0).all()), (name, float(off.max()))  # NaN fails too
