"""LoRA terms of q_proj / v_proj with dropout on the LoRA input, on this repository's fused HIP
products (esep_lora_down / esep_lora_up / esep_lora_grads: the mask regenerated inside them), or
its dropout kernels around vendor-BLAS products for the ranks and sizes that those do not take or
are slower at.

Public API as in the reference's solution/body/lora.py (reference lora.py:140-359):
new_dropout_key, cast_lora_weights, lora_dropout, lora_down_fwd, lora_down_bwd, lora_delta,
lora_up_bwd, LoRAFunction, LoRADeltaFunction, lora_params, lora_forward, with the same
arguments, saved tensors and gradient dtypes.

The term (peft's LoRA Linear under autocast; A [r, in] and B [out, r] without bias):

    term = scaling * (drop(x) @ A^T) @ B^T,   drop(x) = x * keep / (1 - p)

keep is Bernoulli(1 - p) per element of the LoRA input only (the base projection sees the
undropped x); p comes from the peft module and applies only while its nn.Dropout is in
training mode. Every forward call draws a fresh 63-bit key from torch's device generator (no
host sync; torch.manual_seed reproduces it) and the mask is a pure function of (key, element),
so the backward regenerates it from the saved key instead of storing it. The bits differ from
torch's own dropout stream; the law is the same.

Gradients (xa = drop(x) A^T, dterm the incoming gradient):
    dxa = scaling * dterm @ B        dB = scaling * dterm^T @ xa   (fp32)
    dA  = dxa^T @ drop(x)  (fp32)    dx = (dxa @ A) * keep / (1 - p)
Compute dtype: fp16 (the reference's), or bf16 when x is bf16.

LoRAFunction adds the term to the base projection's output (in place when that output is a
fresh dense tensor of the compute dtype: v_proj); LoRADeltaFunction returns the term alone
(q_proj: the RoPE kernel adds it to q, norm_rope.rope(q_delta=...)). Saved for backward by
both: x, xa, the compute-dtype A and B, and the key.
"""

import torch

from . import _hip

_KEY_RANGE = 2 ** 63 - 1


def _compute_dtype(x):
    return torch.bfloat16 if x.dtype == torch.bfloat16 else torch.float16


def new_dropout_key(device):
    """A fresh 63-bit dropout key drawn from torch's generator on `device` (stays there)."""
    return torch.randint(0, _KEY_RANGE, (1,), device=device, dtype=torch.int64)


def cast_lora_weights(weight_a, weight_b, dtype=torch.float16):
    """A and B in the compute dtype, detached (they are r x in and out x r: tiny)."""
    return weight_a.detach().to(dtype), weight_b.detach().to(dtype)


def lora_dropout(x, key, p):
    """x * keep / (1 - p) for a dense 16-bit x, the mask given by `key` (p > 0)."""
    out = torch.empty_like(x)
    _hip.lora_dropout_fwd(x, key, out, p)
    return out


def _fused(rank, *mats):
    """The fused products take this rank and these 16-bit [rows, width] operands: a rank that is a
    multiple of 8 up to 64 (the kernels' tiles; a wider term is an ordinary GEMM, which the
    vendor BLAS runs well), and widths, row strides and addresses of whole 16-byte chunks."""
    if rank % 8 or not 8 <= rank <= 64:
        return False
    for t in mats:
        if not t.is_cuda or t.dim() != 2 or t.dtype not in (torch.float16, torch.bfloat16):
            return False
        rows, width = t.shape
        ld, col = t.stride()
        if (not 0 < rows <= 1 << 22 or width % 8 or not width or col != 1 or ld % 8 or ld < width
                or t.data_ptr() % 16):
            return False
    return True


def _number(scaling):
    """The kernels take the scaling as a number; a tensor (which may be on the graph, or one value per
    column) is torch's to multiply by."""
    return isinstance(scaling, (int, float))


# Where each fused product is the faster one, by rows, width (the long side) and rank, against the
# library's products and the dropout kernels around them: measured on an MI355X for 16 .. 40000 rows,
# widths 64 .. 18944 and ranks 8, 16, 32, 64 in fp16 and bf16 (alike), kernel time of launches back to
# back, library / fused in us. The down kernel's blocks own 16 .. 64 rows and read all of the weight, so
# it loses on wide weights (width x rank) and on few blocks; the gradients' partial sums grow
# with the rank. The term without a base is always the fused kernel's (0.2 .. 0.8 of the library's).


def _down_pays(rows, width, rank, dropout):
    """xa. Without dropout the library reads x once too (rows x width x rank): 4096 x 1536 x 16 5.0 / 4.9,
    5933 x 1536 x 16 5.8 / 7.6, 200 x 8960 x 64 9.9 / 40. With it, the dropout pass is extra: 5933 x 1536
    x 16 26 / 12, but 64 x 8960 x 64 21 / 42 and 40000 x 896 x 64 48 / 61."""
    if dropout:
        return (width <= 2048 or rows >= 1000) if rank <= 32 else width <= 2048 and rows < 8192
    return rows <= 4096 and width * max(rank, 16) <= 32768


def _dxa_pays(rows, width, rank):
    """dxa = scaling * dterm B (two library launches): 5933 x 1536 x 16 8.7 / 6.1, 1000 x 3584 x 16 9.6 / 7.3, but
    2000 x 8960 x 32 21 / 34 and 9000 x 1536 x 64 14 / 20."""
    if width > 2048:
        return width <= 4096 and 32 <= rows <= 2048
    return rank <= 16 or rows < (8192 if rank > 32 else 32768)


def _down_grads_pay(rows, width, rank, dropout, need_dx):
    """dx and dA from one read of x: 5933 x 1536 x 16 29 / 21, with dropout 55 / 26, but 200 x 3584 x 64 11 / 16
    and without dropout 9000 x 8960 x 64 111 / 145. dA alone without dropout is one library product: 4096
    x 1536 x 16 11 / 15, 9000 x 1536 x 16 25 / 18."""
    if not need_dx and not dropout:
        return rows >= 5000 and width <= 4096
    if rank > 32:
        return rows >= 1000 and (dropout or width <= 4096)
    return rank <= 16 or dropout or rows >= 100


def _up_grads_pay(rows, width, rank):
    """dB: 0.3 .. 0.9 of the library up to 4096 wide, but 4096 x 8960 x 16 21 / 27, 4096 x 18944 x 64 42 / 69 and
    64 x 3584 x 64 6.8 / 8.3."""
    if width <= 4096:
        return rank <= 32 or rows >= 450
    return rank <= 16 and rows <= 1000


def _base_pays(rank):
    """base + term, one library product: 4096 x 1536 x 16 10.9 / 7.5 (0.4 .. 1.1 up to rank 16), 9000 x 1536 x 64
    13 / 22 (0.5 .. 1.7 from 32 on)."""
    return rank <= 16


_OUT_DTYPE_OK = True


def _mm_fp32(a, b):
    """a @ b returned in fp32: the BLAS writes fp32 where torch.mm takes out_dtype, else the
    16-bit product is widened (autocast's result)."""
    global _OUT_DTYPE_OK
    if _OUT_DTYPE_OK:
        try:
            return torch.mm(a, b, out_dtype=torch.float32)
        except (RuntimeError, TypeError):
            _OUT_DTYPE_OK = False
    return torch.mm(a, b).float()


def _xa(x, a16, key, p, fused):
    if fused and _down_pays(*x.shape, a16.shape[0], p > 0.0):
        xa = torch.empty((x.shape[0], a16.shape[0]), device=x.device, dtype=x.dtype)
        _hip.lora_down(x, a16, xa, key=key if p > 0.0 else None, p=p)
        return xa
    return torch.mm(lora_dropout(x, key, p) if p > 0.0 else x, a16.t())


def lora_down_fwd(x, a16, key, p):
    """xa = drop(x) @ A^T for a dense x [T, in] (no dropout when p == 0)."""
    return _xa(x, a16, key, p, not _hip.recorded(x, a16) and _fused(a16.shape[0], x, a16)
               and x.is_contiguous() and a16.is_contiguous())


def _dense(t, like):
    return (t.dtype == like.dtype and t.shape == like.shape and t.is_contiguous()
            and t.data_ptr() % 16 == 0)


def _grads_fused(x, a16, dxa):
    return (_fused(a16.shape[0], x, a16, dxa) and x.is_contiguous() and a16.is_contiguous()
            and dxa.is_contiguous())


def _up_bwd_fused(dout, xa, b16):
    """The fused dxa and dB take dout (any row stride), xa and B."""
    return (_fused(b16.shape[1], dout, xa, b16) and xa.is_contiguous() and b16.is_contiguous()
            and dout.dtype == xa.dtype == b16.dtype)


def _dxa(dout, b16, scaling, fused):
    if fused and _dxa_pays(*dout.shape, b16.shape[1]):
        dxa = torch.empty((dout.shape[0], b16.shape[1]), device=dout.device, dtype=dout.dtype)
        _hip.lora_down(dout, b16, dxa, scale=scaling, w_kr=True)
        return dxa
    return torch.mm(dout, b16).mul_(scaling)


def lora_down_bwd(x, a16, dxa, key, p, need_dx=True, dx_accum=None):
    """Backward of lora_down_fwd: (dx or None, dA fp32 [r, in]). With dx_accum (a dense
    [T, in] buffer, e.g. the base projection's dx) the LoRA part of dx is added into it in
    place and it is returned as dx."""
    if (not _hip.recorded(x, a16, dxa, dx_accum) and _grads_fused(x, a16, dxa)
            and _down_grads_pay(*x.shape, a16.shape[0], p > 0.0, need_dx)
            and (not need_dx or dx_accum is None or _dense(dx_accum, x))):
        dx = None
        if need_dx:
            dx = torch.empty_like(x) if dx_accum is None else dx_accum
        da = torch.empty(a16.shape, device=x.device, dtype=torch.float32)
        _hip.lora_grads(x=x, a=a16, dxa=dxa, key=key if p > 0.0 else None, p=p, dx=dx,
                        accumulate=dx_accum is not None, da=da)
        return dx, da
    if not need_dx:
        dropped = lora_dropout(x, key, p) if p > 0.0 else x
        return None, _mm_fp32(dxa.t(), dropped)
    if p == 0.0:
        dx = torch.mm(dxa, a16) if dx_accum is None else dx_accum.addmm_(dxa, a16)
        return dx, _mm_fp32(dxa.t(), x)
    # one kernel pass: the regenerated dropped input (for dA) and the masked, scaled dx,
    # written over the product itself unless it accumulates into dx_accum
    g = torch.mm(dxa, a16)
    dropped = torch.empty_like(x)
    dx = g if dx_accum is None else dx_accum
    _hip.lora_dropout_bwd(x, g, key, dropped, dx, p, accumulate=dx_accum is not None)
    return dx, _mm_fp32(dxa.t(), dropped)


def lora_delta(xa, b16, scaling):
    """The term scaling * xa @ B^T on its own."""
    if (_number(scaling) and not _hip.recorded(xa, b16) and _fused(b16.shape[1], xa, b16)
            and xa.is_contiguous() and b16.is_contiguous() and b16.shape[0] % 8 == 0):
        term = torch.empty((xa.shape[0], b16.shape[0]), device=xa.device, dtype=xa.dtype)
        _hip.lora_up(xa, b16, term, scaling)
        return term
    term = torch.mm(xa, b16.t())
    return term.mul_(scaling)


def lora_up_bwd(dout, xa, b16, scaling):
    """(dxa [T, r], dB fp32 [out, r]) for the term's gradient dout."""
    fused = (_number(scaling) and not _hip.recorded(dout, xa, b16)
             and _up_bwd_fused(dout, xa, b16))
    if fused and _up_grads_pay(*dout.shape, b16.shape[1]):
        db = torch.empty(b16.shape, device=dout.device, dtype=torch.float32)
        _hip.lora_grads(dterm=dout, xa=xa, scale=scaling, db=db)
    else:
        db = _mm_fp32(dout.t(), xa).mul_(scaling)
    return _dxa(dout, b16, scaling, fused), db


def _rows(t, dtype):
    """t [..., k] as a dense [rows, k] tensor of dtype."""
    flat = t.reshape(-1, t.shape[-1])
    return flat.to(dtype).contiguous() if flat.dtype != dtype else flat.contiguous()


def _rows_mm(t, dtype):
    """t [..., k] as a [rows, k] matrix of dtype for torch's products, which take a row stride:
    a 2-D view with unit column stride (such as a column block of a wider gradient) is used as
    it is, anything else as _rows gives it."""
    if t.dim() == 2 and t.dtype == dtype and t.stride(1) == 1 and t.stride(0) >= t.shape[1]:
        return t
    return _rows(t, dtype)


class _LoRATerm:
    """The parts both Functions share: set up the forward (compute dtype, casts, key, xa) and
    turn the term's gradient into (dx, dA, dB) in the dtypes autograd expects. ctx.fused: the
    fused products take x, the rank and the output width (everything between them is dense)."""

    @staticmethod
    def begin(ctx, x, weight_a, weight_b, p, scaling, base=None):
        dtype = _compute_dtype(x)
        x2 = _rows(x, dtype)
        a16, b16 = cast_lora_weights(weight_a, weight_b, dtype)
        key = new_dropout_key(x2.device) if p > 0.0 else None
        ctx.fused = (_number(scaling) and not _hip.recorded(x2, a16, b16, base)
                     and _fused(a16.shape[0], x2, a16, b16) and a16.is_contiguous()
                     and b16.is_contiguous() and b16.shape[0] % 8 == 0)
        xa = _xa(x2, a16, key, p, True) if ctx.fused else lora_down_fwd(x2, a16, key, p)
        ctx.save_for_backward(x2, xa, a16, b16, key)
        ctx.p, ctx.scaling, ctx.dtype = p, scaling, dtype
        ctx.x_shape, ctx.x_dtype = x.shape, x.dtype
        ctx.a_dtype, ctx.b_dtype = weight_a.dtype, weight_b.dtype
        return xa, b16

    @staticmethod
    def grads(ctx, dterm, x_index, a_index):
        x2, xa, a16, b16, key = ctx.saved_tensors
        need = ctx.needs_input_grad
        dt2 = _rows_mm(dterm, ctx.dtype)
        rank, dropout = b16.shape[1], ctx.p > 0.0
        # torch's products for a pass with create_graph, under vmap (is_grads_batched), with a tangent; of
        # the saved tensors only x2 can be on the graph (ctx.fused: none is a wrapper or a subclass)
        if (ctx.fused and not _hip.recorded(dt2, x2) and _hip.dense16(x2, xa, a16, b16)
                and _fused(rank, dt2) and _up_grads_pay(*dt2.shape, rank)
                and _down_grads_pay(*x2.shape, rank, dropout, need[x_index])):
            # dx, dA and dB in one launch after dxa
            dxa = _dxa(dt2, b16, ctx.scaling, True)
            dx = torch.empty_like(x2) if need[x_index] else None
            da = torch.empty(a16.shape, device=x2.device, dtype=torch.float32)
            db = torch.empty(b16.shape, device=x2.device, dtype=torch.float32)
            _hip.lora_grads(x=x2, a=a16, dxa=dxa, key=key, p=ctx.p, dx=dx, da=da, dterm=dt2,
                            xa=xa, scale=ctx.scaling, db=db)
        else:
            dxa, db = lora_up_bwd(dt2, xa, b16, ctx.scaling)
            dx, da = lora_down_bwd(x2, a16, dxa, key, ctx.p, need_dx=need[x_index])
        if dx is not None and (dx.shape != ctx.x_shape or dx.dtype != ctx.x_dtype):
            dx = dx.view(ctx.x_shape).to(ctx.x_dtype)
        return (dx, da.to(ctx.a_dtype) if need[a_index] else None,
                db.to(ctx.b_dtype) if need[a_index + 1] else None)


class LoRAFunction(torch.autograd.Function):
    """apply(x, base, weight_a, weight_b, p, scaling) -> base + term. The term is added into
    base's own buffer when base is a fresh dense (non-view) tensor of the compute dtype (it is
    then marked dirty); otherwise a new tensor is returned."""

    @staticmethod
    def forward(ctx, x, base, weight_a, weight_b, p, scaling):
        xa, b16 = _LoRATerm.begin(ctx, x, weight_a, weight_b, p, scaling, base)
        ctx.base_dtype = base.dtype
        if base.dtype == ctx.dtype and base.is_contiguous() and not base._is_view():
            flat = base.view(-1, base.shape[-1])
            if ctx.fused and _base_pays(b16.shape[1]) and _fused(b16.shape[1], flat):
                _hip.lora_up(xa, b16, flat, scaling, base=flat)
            else:
                flat.addmm_(xa, b16.t(), alpha=scaling)
            ctx.mark_dirty(base)
            return base
        flat = base.reshape(-1, base.shape[-1]).to(ctx.dtype)
        if ctx.fused and _base_pays(b16.shape[1]) and _fused(b16.shape[1], flat):
            out = torch.empty(flat.shape, device=flat.device, dtype=flat.dtype)
            _hip.lora_up(xa, b16, out, scaling, base=flat)
            return out.view(base.shape)
        return torch.addmm(flat, xa, b16.t(), alpha=scaling).view(base.shape)

    @staticmethod
    def backward(ctx, dout):
        dx, da, db = _LoRATerm.grads(ctx, dout, 0, 2)
        dbase = dout.to(ctx.base_dtype) if ctx.needs_input_grad[1] else None
        return dx, dbase, da, db, None, None


class LoRADeltaFunction(torch.autograd.Function):
    """apply(x, weight_a, weight_b, p, scaling) -> term alone, shaped [..., out]; its gradient
    is the gradient of q before the rotation (the RoPE kernel adds the term to q)."""

    @staticmethod
    def forward(ctx, x, weight_a, weight_b, p, scaling):
        xa, b16 = _LoRATerm.begin(ctx, x, weight_a, weight_b, p, scaling)
        if ctx.fused:
            term = torch.empty((xa.shape[0], b16.shape[0]), device=xa.device, dtype=xa.dtype)
            _hip.lora_up(xa, b16, term, scaling)
        else:
            term = lora_delta(xa, b16, scaling)
        return term.view(*x.shape[:-1], term.shape[-1])

    @staticmethod
    def backward(ctx, dterm):
        dx, da, db = _LoRATerm.grads(ctx, dterm, 0, 1)
        return dx, da, db, None, None


def _dropout_p(drop):
    """The dropout probability in effect for a peft LoRA dropout module, or None when it is a
    module this path does not implement."""
    if isinstance(drop, torch.nn.Identity):
        return 0.0
    if isinstance(drop, torch.nn.Dropout):
        return float(drop.p) if drop.training else 0.0
    return None


def _single_plain_adapter(module, adapter):
    """The adapter is the only active one, present, unmerged, enabled, not a DoRA / variant."""
    if getattr(module, "disable_adapters", False) or getattr(module, "merged", False):
        return False
    if list(getattr(module, "active_adapters", [adapter])) != [adapter]:
        return False
    if adapter not in module.lora_A or adapter in getattr(module, "lora_variant", {}):
        return False
    return not getattr(module, "use_dora", {}).get(adapter, False)


def lora_params(module, adapter="default"):
    """(A weight, B weight, dropout p in effect, scaling) of a peft LoRA layer, or None when the
    layer uses something this path does not implement: a bias on A or B, DoRA or another
    variant, several active adapters, a merged or disabled adapter, a dropout other than
    nn.Dropout / nn.Identity, p >= 1, or a scaling that is not a plain number
    (reference lora.py:319-343)."""
    if not _single_plain_adapter(module, adapter):
        return None
    down, up = module.lora_A[adapter], module.lora_B[adapter]
    if down.bias is not None or up.bias is not None:
        return None
    p = _dropout_p(module.lora_dropout[adapter])
    scale = module.scaling[adapter]
    if p is None or p >= 1.0 or isinstance(scale, bool) or not isinstance(scale, (int, float)):
        return None
    return down.weight, up.weight, p, float(scale)


def lora_forward(module, x, base_out, adapter="default"):
    """base_out + the LoRA term of a peft LoRA layer for input x (base_out, the base
    projection's fresh output, is updated in place when it can be); None when the layer or
    the input is not supported (the caller then runs peft's own forward)."""
    params = lora_params(module, adapter)
    if params is None or not x.is_cuda:
        return None
    weight_a, weight_b, p, scaling = params
    return LoRAFunction.apply(x, base_out, weight_a, weight_b, p, scaling)
