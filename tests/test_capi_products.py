"""Argument checks of the product entries (LoRA, GEMM) and of the LM head's row entries, without a
GPU: a bad argument is refused with a negative status and a message before anything is launched,
and the workspace sizes and the GEMM's rule answer for every size without a device."""

import pytest

from solution.body import _hip

A = 256  # stands for an aligned device address; refused calls never read it


def _call(name, base, kw):
    args = dict(base)
    assert set(kw) <= set(args), kw
    args.update(kw)
    return getattr(_hip.lib(), name)(*args.values())


DOWN = dict(x=A, ld_x=64, w=A, w_kr=0, key=A, p=0.1, scale=1.0, out=A, T=4, K=64, r=8, dt=1, s=None)
UP = dict(xa=A, b=A, base=A, ld_base=64, out=A, ld_out=64, scale=1.0, T=4, N=64, r=8, dt=2, s=None)
GRADS = dict(x=A, a=A, dxa=A, key=A, p=0.1, dx=A, acc=0, da=A, dterm=A, ld_dterm=64, xa=A, scale=1.0,
             db=A, ws=A, T=4, K=64, N=64, r=8, dt=1, s=None)
GEMM = dict(a=A, lda=64, b=A, ldb=64, b_kn=0, bias=None, c=A, ldc=64, c_dt=1, ws=A, M=4, N=64, K=64,
            dt=1, s=None)
PART = dict(target=A, cew=A, N=4, V=8, perm=A, inv=A, n_live=A, s=None)
LOSS = dict(target=A, cew=A, ce=A, N=4, V=8, loss=A, s=None)
DX = dict(prod=A, n_live=2, inv=A, cew=A, dloss=A, g_scale=1024.0, dx=A, dx_dt=1, N=4, H=64, s=None)
EINVAL, ESHAPE, EALIGN = -1, -2, -3


@pytest.mark.parametrize("name,base,kw,status", [
    ("esep_lora_down", DOWN, dict(dt=0), EINVAL), ("esep_lora_down", DOWN, dict(r=4), ESHAPE),
    ("esep_lora_down", DOWN, dict(r=12), ESHAPE), ("esep_lora_down", DOWN, dict(r=1 << 20), ESHAPE),
    ("esep_lora_down", DOWN, dict(K=60), ESHAPE), ("esep_lora_down", DOWN, dict(ld_x=56), ESHAPE),
    ("esep_lora_down", DOWN, dict(ld_x=66), ESHAPE), ("esep_lora_down", DOWN, dict(T=-1), ESHAPE),
    ("esep_lora_down", DOWN, dict(p=1.0), EINVAL), ("esep_lora_down", DOWN, dict(p=0.0), EINVAL),
    ("esep_lora_down", DOWN, dict(w_kr=1), EINVAL), ("esep_lora_down", DOWN, dict(w=None), EINVAL),
    ("esep_lora_down", DOWN, dict(x=A + 8), EALIGN), ("esep_lora_down", DOWN, dict(key=A + 4), EALIGN),
    ("esep_lora_down", DOWN, dict(T=0, x=None), 0),
    ("esep_lora_up", UP, dict(dt=3), EINVAL), ("esep_lora_up", UP, dict(N=0), ESHAPE),
    ("esep_lora_up", UP, dict(ld_out=60), ESHAPE), ("esep_lora_up", UP, dict(ld_base=32), ESHAPE),
    ("esep_lora_up", UP, dict(out=None), EINVAL), ("esep_lora_up", UP, dict(base=A + 2), EALIGN),
    ("esep_lora_up", UP, dict(T=0), 0),
    ("esep_lora_grads", GRADS, dict(x=None, dterm=None), EINVAL),
    ("esep_lora_grads", GRADS, dict(da=None), EINVAL), ("esep_lora_grads", GRADS, dict(a=None), EINVAL),
    ("esep_lora_grads", GRADS, dict(xa=None), EINVAL), ("esep_lora_grads", GRADS, dict(ld_dterm=32), EINVAL),
    ("esep_lora_grads", GRADS, dict(p=1.5), EINVAL), ("esep_lora_grads", GRADS, dict(T=0), ESHAPE),
    ("esep_lora_grads", GRADS, dict(ws=None), EINVAL), ("esep_lora_grads", GRADS, dict(dx=A + 8), EALIGN),
    ("esep_gemm", GEMM, dict(dt=0, c_dt=0), EINVAL), ("esep_gemm", GEMM, dict(c_dt=2), EINVAL),
    ("esep_gemm", GEMM, dict(K=96, lda=96, ldb=96), ESHAPE), ("esep_gemm", GEMM, dict(N=60), ESHAPE),
    ("esep_gemm", GEMM, dict(M=0), ESHAPE), ("esep_gemm", GEMM, dict(lda=56), ESHAPE),
    ("esep_gemm", GEMM, dict(ldb=68), ESHAPE), ("esep_gemm", GEMM, dict(ldc=32), ESHAPE),
    ("esep_gemm", GEMM, dict(lda=1 << 23), ESHAPE), ("esep_gemm", GEMM, dict(b=None), EINVAL),
    ("esep_gemm", GEMM, dict(bias=A, c_dt=0), EINVAL), ("esep_gemm", GEMM, dict(c=A + 8), EALIGN),
    ("esep_gemm", GEMM, dict(bias=A + 2), EALIGN),
    ("esep_head_partition", PART, dict(N=0), ESHAPE), ("esep_head_partition", PART, dict(N=1 << 31), ESHAPE),
    ("esep_head_partition", PART, dict(n_live=None), EINVAL),
    ("esep_head_loss", LOSS, dict(V=0), ESHAPE), ("esep_head_loss", LOSS, dict(ce=None), EINVAL),
    ("esep_head_dx", DX, dict(dx_dt=7), EINVAL), ("esep_head_dx", DX, dict(H=60), ESHAPE),
    ("esep_head_dx", DX, dict(n_live=5), ESHAPE), ("esep_head_dx", DX, dict(prod=None), EINVAL),
    ("esep_head_dx", DX, dict(N=1 << 29, H=64), ESHAPE), ("esep_head_dx", DX, dict(N=1 << 62), ESHAPE),
    ("esep_head_dx", DX, dict(g_scale=0.0), EINVAL), ("esep_head_dx", DX, dict(dx=A + 4), EALIGN),
])
def test_arguments_are_refused(name, base, kw, status):
    assert _call(name, base, kw) == status
    if status:
        assert _hip.lib().esep_last_error().startswith(name[len("esep_"):].encode())


def test_gemm_plan_bounds():
    """A product that is taken leaves at least 14 slabs of 64 to its contraction (K >= 896), and its
    partial sums stay within 2^26 floats: whole multiples of the output, at least two of them."""
    lib = _hip.lib()
    for M in (1, 8, 100, 257, 1031, 4096, 30000):
        for N in (8, 136, 1536, 8960, 152064):
            for K in (64, 832, 896, 1536, 17920, 151936):
                ws = lib.esep_gemm_workspace(M, N, K)
                assert ws == 0 or (ws % (M * N) == 0 and ws // (M * N) >= 2 and ws <= 1 << 26), (M, N, K)
                for kn in (0, 1):
                    if lib.esep_gemm_pays(M, N, K, kn):
                        assert K >= 896, (M, N, K)
    assert lib.esep_gemm_pays(1031, 1536, 17920, 1) == 1  # few tiles, long contraction
    assert lib.esep_gemm_plan(1031, 1536, 17950) == ESHAPE and lib.esep_gemm_plan(1, 8, 64) == 4 | 1 << 4
    assert lib.esep_gemm_pays(1031, 1536, 17950, 1) == 0 and lib.esep_gemm_workspace(4, 60, 64) == 0
    assert lib.esep_lora_grads_workspace(0, 64, 64, 8) == 0
    assert lib.esep_lora_grads_workspace(100, 64, 128, 16) % (16 * (64 + 128)) == 0
