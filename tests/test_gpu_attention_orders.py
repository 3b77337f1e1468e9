"""The block orders of the attention kernels (csrc/attention.hpp, attn_order): every order runs the same
blocks, so results are the same bits whichever a launch takes; and max_seqlen is any bound, whose
slack costs little."""

import pytest
import torch

from _util import DEV

pytestmark = pytest.mark.gpu


def _inputs(T, hq, hk, D, dtype=torch.bfloat16, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed + T + D)
    q, do = (torch.randn(T, hq, D, generator=g, device=DEV).to(dtype) for _ in range(2))
    k, v = (torch.randn(T, hk, D, generator=g, device=DEV).to(dtype) for _ in range(2))
    return q, k, v, do


def _run(ins, lens, bound):
    from solution.body import _hip
    from solution.body.attention import cu_seqlens_from_lengths

    q, k, v, do = ins
    o, lse = torch.zeros_like(q), torch.zeros(q.shape[1], q.shape[0], device=DEV)
    dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
    cu, scale = cu_seqlens_from_lengths(lens, DEV), q.shape[2] ** -0.5
    _hip.attn_fwd(q, k, v, o, cu, bound, scale, lse=lse)
    _hip.attn_bwd(q, k, v, o, do, lse, dq, dk, dv, cu, bound, scale)
    return o, lse, dq, dk, dv


GROUPS, TILES, SORTED, LEVEL = range(4)
RAGGED, ALIKE = [129, 1, 0, 700, 257], [300 + i for i in range(16)]
MANY = [100 + 37 * i % 200 for i in range(70)]
# lens, heads, then per bound the expected orders of (forward, dQ, dK / dV) at D = 64 and at D = 128: a block
# per CU at most; a few rounds of blocks; more rounds than the forward and dQ, then than dK / dV take
# longest first; several reversed runs of 256 blocks; sequences of one length; past 64 sequences
CASES = [
    (RAGGED, 4, 2, {700: ((GROUPS,) * 3, (GROUPS,) * 3), 5000: ((LEVEL,) * 3, (LEVEL,) * 3),
                    30000: ((SORTED, SORTED, LEVEL),) * 2, 50000: ((SORTED,) * 3,) * 2}),
    (ALIKE, 12, 12, {315: ((LEVEL,) * 3, (TILES,) * 3), 400: ((LEVEL,) * 3,) * 2,
                     3000: ((SORTED, SORTED, LEVEL),) * 2}),
    (MANY, 4, 4, {299: ((TILES,) * 3,) * 2, 4000: ((GROUPS,) * 3,) * 2}),
]


def _orders(lens, hq, hk, D, bound):
    from solution.body import _hip

    code = _hip.lib().esep_attn_orders(sum(lens), hq, hk, D, len(lens), bound)
    assert code >= 0
    return code & 15, code >> 4 & 15, code >> 8


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("lens,hq,hk,bounds", CASES, ids=["ragged", "alike", "many"])
def test_every_order_gives_the_same_bits(lens, hq, hk, bounds, D):
    ins, want = _inputs(sum(lens), hq, hk, D), None
    for bound, orders in bounds.items():
        assert _orders(lens, hq, hk, D, bound) == orders[D == 128], bound
        got = _run(ins, lens, bound)
        want = want or got
        for a, b in zip(got, want):
            assert torch.equal(a, b), bound
    # and against each sequence on its own (the forward and dQ; dK / dV's sums are split by the shape)
    t0 = 0
    for n in lens[:6]:
        one = [t[t0:t0 + n].contiguous() for t in ins]
        if n:
            o, _, dq, _, _ = _run(one, [n], n)
            assert torch.equal(o, want[0][t0:t0 + n]) and torch.equal(dq, want[2][t0:t0 + n])
        t0 += n


@pytest.mark.parametrize("D,order", [(64, LEVEL), (128, TILES)])
def test_sequences_past_the_bound(D, order):
    """A bound below the longest sequence (not a supported call, but in bounds): the grid holds two
    tiles per sequence, the last ones of the forward and dQ, and nothing else is written."""
    lens = [700] * 12
    ins = _inputs(sum(lens), 16, 16, D)
    assert _orders(lens, 16, 16, D, 256)[:2] == (order, order)
    want, got = _run(ins, lens, 700), _run(ins, lens, 256)
    for i in (0, 2):  # o, dq: query tiles 4 and 5 of 6
        for t0 in range(0, sum(lens), 700):
            assert torch.equal(got[i][t0 + 512:t0 + 700], want[i][t0 + 512:t0 + 700])
            assert not bool(got[i][t0:t0 + 512].any())


@pytest.mark.parametrize("D", [64, 128])
def test_a_loose_bound_costs_little(D):
    """One sequence of 100 tokens under a bound of 65536: the grid's other blocks leave at once (D = 64
    forward 5 us under either bound; a walk over the bound's tiles in each block took 151). Graphs of
    20 launches, so that the host's time does not count."""
    from solution.body import _hip
    from solution.body.attention import cu_seqlens_from_lengths

    q, k, v, do = _inputs(100, 1, 1, D)
    o, lse, cu = torch.empty_like(q), torch.empty(1, 100, device=DEV), cu_seqlens_from_lengths([100], DEV)
    dq, dk, dv = (torch.empty_like(t) for t in (q, k, v))

    def us(bound):
        def launch():
            _hip.attn_fwd(q, k, v, o, cu, bound, 0.125, lse=lse)
            _hip.attn_bwd(q, k, v, o, do, lse, dq, dk, dv, cu, bound, 0.125)

        launch()
        torch.cuda.synchronize()
        graph, best = torch.cuda.CUDAGraph(), float("inf")
        with torch.cuda.graph(graph):
            for _ in range(20):
                launch()
        for _ in range(6):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            graph.replay()
            end.record()
            torch.cuda.synchronize()
            best = min(best, start.elapsed_time(end) / 20 * 1e3)
        return best

    tight, loose = us(128), us(65536)
    assert loose < 3 * tight, (tight, loose)


@pytest.mark.parametrize("D", [64, 128])
def test_more_blocks_than_one_grid_dimension_holds(D):
    """20000 short sequences under a loose bound: 17.9 million blocks, where HIP takes fewer than 2^32
    threads (2^24 blocks) per grid dimension."""
    lens = [1 + i % 8 for i in range(20000)]
    ins = _inputs(sum(lens), 14, 2, D)
    for a, b in zip(_run(ins, lens, 8192), _run(ins, lens, 8)):
        assert torch.equal(a, b)
