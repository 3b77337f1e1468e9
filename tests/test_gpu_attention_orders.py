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


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("lens,bounds", [([100], (128, 4097, 65536)),
                                         ([129, 1, 0, 700, 257], (700, 1000, 5000)),
                                         ([200] * 12, (200, 1024, 8192))])
def test_any_bound_gives_the_same_bits(lens, bounds, D):
    ins = _inputs(sum(lens), 4, 2, D)
    want = _run(ins, lens, max(lens))
    for bound in bounds:
        for a, b in zip(_run(ins, lens, bound), want):
            assert torch.equal(a, b), bound


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
