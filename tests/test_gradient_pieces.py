"""Backward kernels whose sums are dealt to several workgroups (``FA_PIECES``) and the kernel that adds their fp32
slices: on the simulator against the same kernels in one piece, on the GPU through the public operator at shapes whose
launches would leave the device half empty, against the oracle."""
import math

import pytest
import torch

import flag_attn
from flagattention_amd import _abi
from oracle import flash_attention as oracle_flash, within_two_x
from tests.sim import simlib


@pytest.mark.parametrize("B,H,Hk,M,N,D,causal,pieces", [
    (1, 2, 2, 200, 260, 64, True, 3),       # fewer tiles than pieces under the mask: some are empty
    (2, 2, 1, 330, 130, 128, True, 2),      # rows without keys, two heads per kv head
    (1, 1, 1, 70, 65, 16, False, 4),        # two tiles, four pieces
    (1, 2, 2, 257, 190, 32, False, 2),
])
def test_pieces_add_up_on_the_simulator(B, H, Hk, M, N, D, causal, pieces):
    lib, scale = simlib.get(), 1 / math.sqrt(D)
    g = torch.Generator().manual_seed(3)
    q, k, v, do = (torch.randn(B, h, t, D, generator=g).to(torch.bfloat16) for h, t in ((H, M), (Hk, N), (Hk, N), (H, M)))
    o, lse, delta = torch.empty_like(q), torch.empty(B, H, M), torch.empty(B, H, M)
    _abi.fa_fwd(lib, q, k, v, o, lse, causal, scale)
    _abi.fa_bwd_delta(lib, o, do, delta)
    ds = torch.full((lib.fa_bwd_ds_workspace_mib(B, H, M, N) << 19,), float("nan"), dtype=torch.bfloat16)
    results = []
    for n in (0, pieces):
        kind = dict(dtype=torch.float32) if n else dict(dtype=torch.bfloat16)
        dk, dv = (torch.full((B, H * max(1, n), N, D), float("nan"), **kind) for _ in range(2))
        dk2, dv2 = torch.full_like(dk, float("nan")), torch.full_like(dv, float("nan"))
        dq, dq2 = (torch.full((B, H * max(1, n), M, D), float("nan"), **kind) for _ in range(2))
        _abi.fa_bwd_dkdv(lib, q, k, v, do, lse, delta, dk, dv, causal, scale, pieces=n)
        _abi.fa_bwd_dq(lib, q, k, v, do, lse, delta, dq, causal, scale, pieces=n)
        _abi.fa_bwd_dkdv_ds(lib, q, k, v, do, lse, delta, dk2, dv2, ds, causal, scale, pieces=n)
        _abi.fa_bwd_dq_from_ds(lib, k, ds, dq2, causal, scale, pieces=n)
        assert torch.equal(dk, dk2) and torch.equal(dv, dv2)
        if n:
            sums = [torch.full((B, H, t, D), float("nan"), dtype=torch.bfloat16) for t in (N, N, M)]
            _abi.fa_sum_slices(lib, (dk, dv, dq), sums)
            sums.append(torch.full_like(sums[2], float("nan")))
            _abi.fa_sum_slices(lib, (dq2,), (sums[3],))
        else:
            sums = [dk, dv, dq, dq2]
        results.append(sums)
    for name, whole, parts in zip(("dk", "dv", "dq", "dq from dS"), *results):
        # the same products, each fp32 sum in another order, rounded once to bf16
        assert (whole.float() - parts.float()).abs().max() <= 2 ** -7 * whole.float().abs().max(), name


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Hk,M,N,D,causal,dtype", [
    (1, 4, 4, 2000, 2000, 64, True, torch.float16),
    (1, 2, 2, 2500, 1300, 32, True, torch.bfloat16),     # rows without keys
    (1, 2, 2, 1100, 3001, 128, True, torch.bfloat16),    # dS kept
    (1, 8, 2, 1111, 1500, 128, False, torch.float16),    # four heads per kv head
    (3, 2, 1, 700, 2000, 16, False, torch.bfloat16),
])
def test_gradients_of_small_launches(B, H, Hk, M, N, D, causal, dtype):
    g = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn(B, h, t, D, dtype=dtype, device="cuda", generator=g).requires_grad_() for h, t in ((H, M), (Hk, N), (Hk, N)))
    do = torch.randn(B, H, M, D, dtype=dtype, device="cuda", generator=g)
    grads = torch.autograd.grad(flag_attn.flash_attention(q, k, v, causal), (q, k, v), do)
    ref = torch.autograd.grad(oracle_flash(q, k, v, causal, upcast=True), (q, k, v), do)
    same = torch.autograd.grad(oracle_flash(q, k, v, causal, upcast=False), (q, k, v), do)
    for name, h, s, r in zip(("dq", "dk", "dv"), grads, same, ref):
        ok, e_hyp, e_same = within_two_x(h, s, r)
        assert ok, f"{name}: kernel err {e_hyp:.3e} vs same-precision torch err {e_same:.3e}"
