"""NF4 dequantization at the edges of its launches (a block covers 64 scale blocks of one weight, 64
or, from 131072 scale blocks in all, 128 of several): the same bits as the oracle, and as one
launch per weight, and nothing written past the output."""

import numpy as np
import pytest
import torch

from _util import DEV
from oracle import nf4_ref as ref

pytestmark = pytest.mark.gpu


def _weight(nb, seed, dtype):
    """Raw state of nb scale blocks and its device form with a guarded output buffer."""
    rng = np.random.default_rng(seed)
    raw = (rng.integers(0, 256, nb * 32, dtype=np.uint8), rng.integers(0, 256, nb, dtype=np.uint8),
           (rng.random((nb + 255) // 256) * 0.1 + 0.01).astype(np.float32),
           np.sort(rng.standard_normal(256)).astype(np.float32), np.float32(rng.random() * 0.05))
    table = ref.NF4 if seed % 2 else (ref.NF4[::-1] * 0.5).astype(np.float32)
    buf = torch.full((nb * 64 + 64,), 7.0, device=DEV, dtype=dtype)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
           for a in (*raw[:4], np.array([raw[4]], dtype=np.float32), table)]
    return raw, table, dev, buf


def _want(raw, table, dtype):
    """The oracle's formula with the weight's own table: fp32 scale in two roundings, one product,
    one rounding to the output type."""
    packed, absmax, absmax2, code2, offset = raw
    prod = (code2[absmax] * absmax2[np.arange(absmax.size) // 256]).astype(np.float32)
    scale = (prod + offset).astype(np.float32)
    nib = np.stack([packed >> 4, packed & 15], 1).reshape(-1)
    return torch.from_numpy((table[nib] * np.repeat(scale, 64)).astype(np.float32)).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32],
                         ids=["fp16", "bf16", "fp32"])
@pytest.mark.parametrize("nb", [1, 63, 64, 65, 257])
def test_one_weight(nb, dtype):
    from solution.body import _hip

    raw, table, dev, buf = _weight(nb, 1, dtype)
    _hip.nf4_dequant(*dev, buf[:nb * 64].view(nb, 64))
    assert torch.equal(buf[:nb * 64].cpu(), _want(raw, table, dtype))
    assert np.array_equal(_want(raw, table, torch.float32).numpy(),
                          ref.dequantize_nf4(*raw, out_dtype=np.float32).reshape(-1))
    assert (buf[nb * 64:] == 7).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32], ids=["fp16", "fp32"])
@pytest.mark.parametrize("sizes", [(1, 1), (63, 1, 64), (65, 127, 2, 1, 1, 30, 128, 5),
                                   (70000, 61071), (70001, 61071), (131072, 3, 128)])
def test_several_weights(sizes, dtype):
    from solution.body import _hip

    ws = [_weight(nb, 2 + i, dtype) for i, nb in enumerate(sizes)]
    _hip.nf4_dequant_multi([(*dev, buf[:nb * 64].view(nb, 64))
                            for nb, (_, _, dev, buf) in zip(sizes, ws)])
    for nb, (raw, table, dev, buf) in zip(sizes, ws):
        assert torch.equal(buf[:nb * 64].cpu(), _want(raw, table, dtype))
        assert (buf[nb * 64:] == 7).all()


def test_more_units_than_one_grid_dimension_holds():
    """2^30 scale blocks and more: a launch of 2^32 threads, which a grid dimension cannot count
    (34 GB of packed bytes, 137 GB of fp16)."""
    from solution.body import _hip

    nb = (1 << 30) + 1000
    if torch.cuda.mem_get_info()[0] < 200 << 30:
        pytest.skip("needs 200 GB of free GPU memory")
    _, _, (_, _, _, code2, offset, table), _ = _weight(4, 1, torch.float16)
    packed = torch.zeros(nb * 32, device=DEV, dtype=torch.uint8)
    absmax = torch.zeros(nb, device=DEV, dtype=torch.uint8)
    absmax2 = torch.full(((nb + 255) // 256,), 0.25, device=DEV)
    out = torch.zeros(nb, 64, device=DEV, dtype=torch.float16)
    at = torch.tensor([0, 999, (1 << 22), (1 << 29) + 3, nb - 1001, nb - 1], device=DEV)
    g = torch.Generator(device=DEV).manual_seed(1)
    bytes_ = torch.randint(0, 256, (6, 32), generator=g, device=DEV, dtype=torch.uint8)
    packed.view(nb, 32)[at] = bytes_
    absmax[at] = torch.arange(6, device=DEV, dtype=torch.uint8) * 40 + 3
    want = torch.empty(6, 64, device=DEV, dtype=torch.float16)
    _hip.nf4_dequant(bytes_, absmax[at], absmax2[:1], code2, offset, table, want)
    _hip.nf4_dequant(packed, absmax, absmax2, code2, offset, table, out)
    assert torch.equal(out[at], want)
    zero = out[at + torch.tensor([1, 1, 1, 1, 1, -1], device=DEV)]  # neighbours: one value each
    assert bool((zero == zero[0, 0]).all()) and float(zero[0, 0]) != 0
    del packed, out
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32],
                         ids=["fp16", "bf16", "fp32"])
@pytest.mark.parametrize("blocks", [1572863, 1572864, 1572929])
def test_outputs_past_the_caches(blocks, dtype):
    """The stores change at 192 MiB of 16-bit output (1572864 scale blocks): the same bits as decoded in
    pieces, one weight and several, and nothing past the output."""
    from solution.body import _hip

    g = torch.Generator(device=DEV).manual_seed(blocks)
    packed = torch.randint(0, 256, (blocks * 32,), generator=g, device=DEV, dtype=torch.uint8)
    absmax = torch.randint(0, 256, (blocks,), generator=g, device=DEV, dtype=torch.uint8)
    absmax2 = torch.rand((blocks + 255) // 256, generator=g, device=DEV)
    _, _, (_, _, _, code2, offset, table), _ = _weight(4, 1, dtype)
    want = torch.empty(blocks * 64, device=DEV, dtype=dtype)
    step = 1 << 18  # whole groups of 256 scale blocks
    for b in range(0, blocks, step):
        e = min(blocks, b + step)
        _hip.nf4_dequant(packed[32 * b:32 * e], absmax[b:e], absmax2[b // 256:], code2, offset, table,
                         want[64 * b:64 * e])
    for cut in (0, 512 * 1000):
        out = torch.full((blocks * 64 + 64,), 7.0, device=DEV, dtype=dtype)
        parts = [(packed[32 * b:32 * e], absmax[b:e], absmax2[b // 256:], code2, offset, table,
                  out[64 * b:64 * e]) for b, e in ((0, cut), (cut, blocks)) if b < e]
        if cut:
            _hip.nf4_dequant_multi(parts)
        else:
            _hip.nf4_dequant(*parts[0])
        assert torch.equal(out[:-64], want) and bool((out[-64:] == 7).all())
