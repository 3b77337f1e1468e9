"""esep_gemm at the edges of its tiles (rows, columns, the 64-deep contraction steps and the splits of
the contraction), both layouts of B, 16-bit and fp32 results, against float64 products.

Bound, with u the unit roundoff of the stored type (2^-11 fp16, 2^-8 bf16) and S the sum of the
products' magnitudes: one rounding of the result (u |want|) and an fp32 sum of at most 2^15 terms
(1e-5 S)."""

import pytest
import torch

from _util import DEV, gen

pytestmark = pytest.mark.gpu

U = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 0.0}

# (M, N, K): one row and one 8-column chunk, one contraction step; ragged tiles of every shape with and
# without splits of the contraction (several rounds, a ragged last tile, an odd number of steps, many
# splits of few rows)
SIZES = [(1, 8, 64), (65, 264, 704), (130, 136, 128), (16, 1536, 17920), (40, 1096, 4096),
         (1031, 896, 9728), (2300, 8960, 256), (3001, 8960, 192), (1031, 1536, 17920),
         (1285, 1544, 4160), (4096, 1544, 1088), (260, 8200, 1024), (8254, 888, 192),
         (1203, 888, 9728), (1750, 896, 4864)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("b_kn", [False, True], ids=["nk", "kn"])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_gemm(M, N, K, b_kn, dtype):
    from solution.body import _hip

    g = torch.Generator(device=DEV).manual_seed(M + N + K)

    def rnd(*shape):
        return torch.randn(*shape, generator=g, device=DEV).to(dtype)

    a = rnd(M, K + 16)[:, 8:8 + K]  # a column block of wider rows
    b = rnd(K, N) if b_kn else rnd(N, K)
    bias = rnd(N)
    w = b.double() if b_kn else b.double().T
    want, S = a.double() @ w, a.double().abs() @ w.abs()
    for out_dtype, bi in ((dtype, None), (dtype, bias), (torch.float32, None)):
        out = torch.full((M, N), float("nan"), device=DEV, dtype=out_dtype)
        _hip.gemm(a, b, out, b_kn=b_kn, bias=bi)
        ref = want if bi is None else want + bi.double()
        err = (out.double() - ref).abs()
        bound = U[out_dtype] * ref.abs() + 1e-5 * (S + 1)
        assert bool((err <= bound).all()), float((err - bound).max())  # NaN fails too
        again = torch.empty_like(out)
        _hip.gemm(a, b, again, b_kn=b_kn, bias=bi)
        assert torch.equal(out, again)


def test_linear_and_matmul_routes():
    """linear / matmul give the product whichever way they go, and leave what the kernel does not
    take to the vendor BLAS (odd widths, transposed views, float32, autocast to another dtype)."""
    from solution.body import _hip

    g, K = gen(5), 17920
    x = torch.randn(3, 100, K, generator=g).half().to(DEV)
    w = (torch.randn(256, K, generator=g) * 0.01).half().to(DEV)
    b = torch.randn(256, generator=g).half().to(DEV)
    assert _hip.gemm_takes(x.view(-1, K), w, False)
    want = x.double() @ w.double().T + b.double()
    with _hip.count_launches() as names:
        y = _hip.linear(x, w, b)
        dx = _hip.matmul(y.detach(), w)
    assert names == ["_gemm"]  # the 256-deep product is left to the library
    assert y.shape == (3, 100, 256) and dx.shape == x.shape
    # |x| . |w| sums to about 17920 * 0.8 * 0.008
    assert (y.double() - want).abs().max() <= 2.0 ** -11 * want.abs().max() + 1e-5 * 115
    ref = y.double() @ w.double()
    assert (dx.double() - ref).abs().max() <= 2.0 ** -10 * ref.abs().max()
    for xx, ww in ((x[0], w.t().contiguous().t()), (x[0].float(), w.float()), (x[0, :, :K - 1], w[:, :K - 1])):
        assert not _hip.gemm_takes(xx, ww, False)
        assert _hip.linear(xx, ww).shape == (100, 256)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert _hip.linear(x, w).dtype == torch.bfloat16


def test_a_bias_that_broadcasts():
    """F.linear takes biases that broadcast to the output: those are the library's."""
    from solution.body import _hip

    x, w = torch.randn(64, 17920, device=DEV).half(), torch.randn(1024, 17920, device=DEV).half()
    assert _hip.gemm_takes(x, w, False)
    for bias in (torch.randn(1, device=DEV).half(), torch.randn(1, 1024, device=DEV).half()):
        assert torch.equal(_hip.linear(x, w, bias), torch.nn.functional.linear(x, w, bias))
