"""Calls that torch has to see as its own operations (a graph through the public product functions, a
recorded backward pass, forward-mode tangents, vmap and batched gradients) keep them: the fused
kernels fill buffers behind torch's back. Results against the same products written in torch."""

import pytest
import torch
import torch.autograd.forward_ad as fwd

from _util import DEV

pytestmark = pytest.mark.gpu

T, K, N, R, S = 40, 64, 128, 16, 2.0
# products of fp16 operands of up to 128 terms, results rounded once or twice (2^-11 each)
TOL = dict(rtol=4e-3, atol=4e-3)


def _rnd(*shape, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g, device=DEV) * 0.5).half()


def _same(got, want):
    got, want = (t if isinstance(t, tuple) else (t,) for t in (got, want))
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        if a is not None:
            torch.testing.assert_close(a.float(), b.float(), **TOL)


def _ref_delta(xa, b):
    return S * (xa @ b.t())


def _ref_down(x, a):
    return x @ a.t()


def _ref_up_bwd(dout, xa, b):
    return S * (dout @ b), S * (dout.t() @ xa).float()


def _ref_down_bwd(x, a, dxa):
    return dxa @ a, (dxa.t() @ x).float()


def _functions():
    """(function, torch's form, operands); p = 0 throughout."""
    from solution.body import lora as L

    x, a, xa, b, d, dxa = _rnd(T, K), _rnd(R, K), _rnd(T, R), _rnd(N, R), _rnd(T, N), _rnd(T, R, seed=1)
    return {
        "delta": (lambda xa, b: L.lora_delta(xa, b, S), _ref_delta, (xa, b)),
        "down_fwd": (lambda x, a: L.lora_down_fwd(x, a, None, 0.0), _ref_down, (x, a)),
        "up_bwd": (lambda d, xa, b: L.lora_up_bwd(d, xa, b, S), _ref_up_bwd, (d, xa, b)),
        "down_bwd": (lambda x, a, dxa: L.lora_down_bwd(x, a, dxa, None, 0.0), _ref_down_bwd, (x, a, dxa)),
    }


@pytest.fixture(autouse=True)
def _fp32_products(monkeypatch):
    """lora._mm_fp32 gives up torch's out_dtype for good where torch refuses it (forward mode)."""
    from solution.body import lora as L

    monkeypatch.setattr(L, "_OUT_DTYPE_OK", L._OUT_DTYPE_OK)


@pytest.mark.parametrize("name", ["delta", "down_fwd"])
@pytest.mark.parametrize("which", [0, 1])
def test_graph_of_the_forward_products(name, which):
    f, ref, ops = _functions()[name]
    grads = []
    for fn in (f, ref):
        ins = [t.clone().requires_grad_(i == which) for i, t in enumerate(ops)]
        out = fn(*ins)
        grads.append(torch.autograd.grad(out, ins[which], torch.ones_like(out))[0])
    _same(*grads)
    with torch.no_grad():  # the kernels' own result
        _same(f(*ops), ref(*ops))


def test_graph_of_the_dropped_product():
    """With dropout on, the product's other operand still gets its gradient."""
    from solution.body import lora as L

    x, key = _rnd(T, K), torch.tensor([77], device=DEV)
    a = _rnd(R, K).requires_grad_()
    out = L.lora_down_fwd(x, a, key, 0.25)
    (da,) = torch.autograd.grad(out, a, torch.ones_like(out))
    want = torch.ones_like(out).t() @ L.lora_dropout(x, key, 0.25)
    _same(da, want)


def test_scaling_given_as_a_tensor():
    """A scaling on the graph gets its gradient, and one value per column is taken."""
    from solution.body import lora as L

    xa, b, d = _rnd(T, R), _rnd(N, R), _rnd(T, N)
    scale = torch.tensor(S, device=DEV, requires_grad=True)
    out = L.lora_delta(xa, b, scale)
    _same(out.detach(), _ref_delta(xa, b))
    (ds,) = torch.autograd.grad(out, scale, d)
    torch.testing.assert_close(ds, ((xa @ b.t()).float() * d.float()).sum(), rtol=2e-2, atol=2.0)
    columns = torch.rand(N, device=DEV).half()
    _same(L.lora_delta(xa, b, columns), (xa @ b.t()) * columns)
    _same(L.lora_up_bwd(d, xa, b, torch.tensor(S, device=DEV)), _ref_up_bwd(d, xa, b))
    term = L.LoRADeltaFunction.apply(_rnd(T, K), _rnd(R, K), b, 0.0, torch.tensor(S, device=DEV))
    _same(term, S * ((_rnd(T, K) @ _rnd(R, K).t()) @ b.t()))


@pytest.mark.parametrize("name", ["delta", "down_fwd", "up_bwd", "down_bwd"])
def test_traced(name):
    """A trace holds the products themselves: it computes them for other inputs."""
    fn, ref, ops = _functions()[name]
    traced = torch.jit.trace(fn, ops, check_trace=False)
    other = tuple(t.flip(0).contiguous() for t in ops)
    _same(traced(*other), ref(*other))


@pytest.mark.parametrize("name", ["delta", "down_fwd", "up_bwd", "down_bwd"])
def test_seen_by_modes_and_subclasses(name):
    """A dispatch mode sees the products, and a subclass gets its own type back."""
    from torch.utils._python_dispatch import TorchDispatchMode

    class Count(TorchDispatchMode):
        n = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.n += func.overloadpacket is torch.ops.aten.mm
            return func(*args, **(kwargs or {}))

    class Marked(torch.Tensor):
        pass

    fn, ref, ops = _functions()[name]
    with Count() as count:
        got = fn(*ops)
    assert count.n == (2 if name.endswith("bwd") else 1)
    _same(got, ref(*ops))
    marked = fn(*(t.as_subclass(Marked) for t in ops))
    assert all(type(t) is Marked for t in (marked if isinstance(marked, tuple) else (marked,)))


@pytest.mark.parametrize("name", ["delta", "down_fwd", "up_bwd", "down_bwd"])
def test_compiled_and_fake(name):
    from torch._subclasses.fake_tensor import FakeTensorMode

    fn, ref, ops = _functions()[name]
    compiled = torch.compile(fn, backend="eager", fullgraph=True)
    _same(compiled(*ops), ref(*ops))
    with FakeTensorMode() as mode:
        fakes = fn(*(mode.from_tensor(t) for t in ops))
    for f, r in zip(*((t if isinstance(t, tuple) else (t,)) for t in (fakes, ref(*ops)))):
        assert f.shape == r.shape and f.dtype == r.dtype


def test_term_under_a_trace():
    from solution.body import lora as L

    traced = torch.jit.trace(lambda x, a, b: L.LoRADeltaFunction.apply(x, a, b, 0.0, S),
                             (_rnd(T, K), _rnd(R, K), _rnd(N, R)), check_trace=False)
    x, a, b = _rnd(T, K, seed=1), _rnd(R, K, seed=1), _rnd(N, R, seed=1)
    _same(traced(x, a, b), S * ((x @ a.t()) @ b.t()))


@pytest.mark.parametrize("name,which,out", [("up_bwd", 2, 0), ("down_bwd", 1, 0)])
def test_graph_of_the_backward_products(name, which, out):
    """Their 16-bit results are differentiable in every operand, not in the incoming gradient alone."""
    f, ref, ops = _functions()[name]
    grads = []
    for fn in (f, ref):
        ins = [t.clone().requires_grad_(i == which) for i, t in enumerate(ops)]
        o = fn(*ins)[out]
        grads.append(torch.autograd.grad(o, ins[which], torch.ones_like(o))[0])
    _same(*grads)


@pytest.mark.parametrize("name,which", [("up_bwd", 1), ("down_bwd", 0)])
def test_fp32_results_are_on_the_graph(name, which):
    """The fp32 results stand on the graph of an operand that requires grad (torch then says itself
    that it has no derivative for them), instead of passing for constants."""
    f, _, ops = _functions()[name]
    ins = [t.clone().requires_grad_(i == which) for i, t in enumerate(ops)]
    assert f(*ins)[1].requires_grad


@pytest.mark.parametrize("name", ["delta", "down_fwd", "up_bwd", "down_bwd"])
def test_forward_mode(name):
    f, ref, ops = _functions()[name]
    which = len(ops) - 1
    tangents = []
    for fn in (f, ref):
        with fwd.dual_level():
            ins = list(ops)
            ins[which] = fwd.make_dual(ops[which], _rnd(*ops[which].shape, seed=5))
            out = fn(*ins)
            tangents.append(tuple(fwd.unpack_dual(o).tangent
                                  for o in (out if isinstance(out, tuple) else (out,))))
    _same(*tangents)


@pytest.mark.parametrize("name", ["delta", "down_fwd", "up_bwd", "down_bwd"])
@pytest.mark.filterwarnings("ignore:There is a performance drop")
def test_vmap(name):
    f, ref, ops = _functions()[name]
    dims = [None] * len(ops)
    dims[-1] = 0
    ins = (*ops[:-1], torch.stack([ops[-1], -ops[-1], 2 * ops[-1]]))
    _same(torch.vmap(f, tuple(dims))(*ins), torch.vmap(ref, tuple(dims))(*ins))


def _lora_function(name, x, a, b):
    from solution.body import lora as L

    if name == "delta":
        return L.LoRADeltaFunction.apply(x, a, b, 0.0, S)
    return L.LoRAFunction.apply(x, torch.zeros(T, N, device=DEV).half(), a, b, 0.0, S)


@pytest.mark.parametrize("name", ["delta", "added"])
@pytest.mark.filterwarnings("ignore:There is a performance drop")
def test_batched_gradients_of_the_term(name):
    """torch.autograd.grad(is_grads_batched=True) runs the backward pass under vmap."""
    ops = [t.clone().requires_grad_() for t in (_rnd(T, K), _rnd(R, K).float(), _rnd(N, R).float())]
    out = _lora_function(name, *ops)
    d = torch.stack([_rnd(T, N), _rnd(T, N, seed=3)])
    got = torch.autograd.grad(out, ops, d, is_grads_batched=True, retain_graph=True)
    for i in range(2):
        want = torch.autograd.grad(out, ops, d[i], retain_graph=True)
        _same(tuple(g[i] for g in got), want)


@pytest.mark.parametrize("name", ["delta", "added"])
def test_tangent_of_the_incoming_gradient(name):
    ops = [t.clone().requires_grad_() for t in (_rnd(T, K), _rnd(R, K).float(), _rnd(N, R).float())]
    out = _lora_function(name, *ops)
    d, t = _rnd(T, N), _rnd(T, N, seed=3)
    with fwd.dual_level():
        got = torch.autograd.grad(out, ops, fwd.make_dual(d, t), retain_graph=True)
        got = tuple(fwd.unpack_dual(g).tangent for g in got)
    _same(got, torch.autograd.grad(out, ops, t))  # the backward pass is linear in it


def test_recorded_pass_over_a_constant_gradient():
    """create_graph with an incoming gradient that is a constant: what the backward pass computes from
    tensors on the graph is on it."""
    ops = [t.clone().requires_grad_() for t in (_rnd(T, K), _rnd(R, K).float(), _rnd(N, R).float())]
    out = _lora_function("delta", *ops)
    _, da, _ = torch.autograd.grad(out, ops, torch.ones_like(out), create_graph=True)
    assert da.requires_grad  # dA is a product with x


class _State:
    """A quant state of random NF4 bytes [n, k]."""

    def __init__(self, n, k):
        g = torch.Generator(device=DEV).manual_seed(n + k)
        nb = n * k // 64
        self.packed = torch.randint(0, 256, (nb * 32,), generator=g, device=DEV, dtype=torch.uint8)
        self.quant_type, self.blocksize, self.nested, self.shape = "nf4", 64, True, (n, k)
        self.absmax = torch.randint(0, 256, (nb,), generator=g, device=DEV, dtype=torch.uint8)
        self.code = torch.linspace(-1, 1, 16, device=DEV)
        self.offset = torch.tensor(0.02, device=DEV)
        self.state2 = type("S", (), dict(absmax=torch.full(((nb + 255) // 256,), 0.02, device=DEV),
                                         code=torch.linspace(-1, 1, 256, device=DEV), blocksize=256))()


@pytest.mark.parametrize("multi", [False, True])
def test_nf4_backward_under_vmap_and_forward_mode(multi):
    """The NF4 linears' dX where esep_gemm would take it (17920 outputs contracted)."""
    from solution import nf4
    from solution.body import _hip

    st = _State(17920, 64)
    x = _rnd(T, 64).requires_grad_()
    y = (nf4.NF4MultiLinear.apply(x, None, ([st.packed], [st], None)) if multi
         else nf4.nf4_linear(x, st.packed, None, st))
    d = torch.stack([_rnd(T, 17920), _rnd(T, 17920, seed=3)])
    with _hip.count_launches() as names:
        want = [torch.autograd.grad(y, x, di, retain_graph=True)[0] for di in d]
    assert "_gemm" in names
    (got,) = torch.autograd.grad(y, x, d, is_grads_batched=True, retain_graph=True)
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=4e-3, atol=1e-2)  # |dX| about 0.5, two kernels
    with fwd.dual_level():
        (dx,) = torch.autograd.grad(y, x, fwd.make_dual(d[0], d[1]), retain_graph=True)
        torch.testing.assert_close(fwd.unpack_dual(dx).tangent, want[1], rtol=4e-3, atol=1e-2)


def test_linear_and_matmul_see_every_operand():
    """A weight or a bias that requires grad in grad mode goes to torch's product too."""
    from solution.body import _hip

    x, w, wk, b = _rnd(T, 17920), _rnd(2048, 17920), _rnd(17920, N), _rnd(2048)
    for t in (w, b):
        t.requires_grad_()
        assert _hip.linear(x, w, b).requires_grad
        t.requires_grad_(False)
    assert _hip.matmul(x, wk.requires_grad_()).requires_grad
    with torch.no_grad(), _hip.count_launches() as names:
        _hip.linear(x, w, b), _hip.matmul(x, wk)
    assert names == ["_gemm", "_gemm"]


def test_head_loss_gradient_batched_and_tangent():
    from solution.head import fused_linear_ce

    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(30, 64, generator=g, device=DEV, requires_grad=True)
    w = (torch.randn(100, 64, generator=g, device=DEV) * 0.1).half()
    target = torch.randint(-5, 100, (30,), generator=g, device=DEV)
    loss, _ = fused_linear_ce(x, w, target, torch.rand(30, generator=g, device=DEV))
    (plain,) = torch.autograd.grad(loss, x, retain_graph=True)
    scale = torch.tensor([1.0, -2.5], device=DEV)
    (got,) = torch.autograd.grad(loss, x, scale, is_grads_batched=True, retain_graph=True)
    torch.testing.assert_close(got, torch.stack([plain, -2.5 * plain]), rtol=1e-6, atol=0)
    with fwd.dual_level():
        (dx,) = torch.autograd.grad(loss, x, fwd.make_dual(scale[0], scale[1]))
        torch.testing.assert_close(fwd.unpack_dual(dx).tangent, -2.5 * plain, rtol=1e-6, atol=0)


def _transposed(t):
    return t.t().contiguous().t() if t.dim() == 2 else t


def _moved(t):
    """The same values at an address that is 8 bytes past a 16-byte one."""
    room = torch.empty(t.numel() + 16 // t.element_size(), device=t.device, dtype=t.dtype)
    return room[8 // t.element_size():][:t.numel()].view(t.shape).copy_(t)


@pytest.mark.parametrize("unpack", [_transposed, _moved])
@pytest.mark.parametrize("what", ["lora", "delta", "head"])
def test_saved_tensors_given_back_otherwise(what, unpack):
    """Saved-tensor hooks may give back other strides and addresses."""
    from solution.body import lora as L
    from solution.head.op import fused_linear_ce

    def run():
        if what == "head":
            x, w = _rnd(T, K).requires_grad_(), _rnd(N, K)
            target = torch.arange(T, device=DEV)
            target[::5] = -100
            out = fused_linear_ce(x, w, target, torch.ones(T, device=DEV), chunk_rows=16)[0]
            return torch.autograd.grad(out, (x,))
        x, a, b = (_rnd(*s).requires_grad_() for s in ((T, K), (R, K), (N, R)))
        if what == "lora":
            out = L.LoRAFunction.apply(x, _rnd(T, N), a, b, 0.0, S)
        else:
            out = L.LoRADeltaFunction.apply(x, a, b, 0.0, S)
        return torch.autograd.grad(out, (x, a, b), _rnd(T, N, seed=2))

    want = run()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        got = run()
    _same(got, want)
