"""Backward kernels whose sums are dealt to several workgroups (``FA_PIECES``) and the kernel that adds their fp32
slices: on the simulator against the same kernels in one piece, on the GPU through the public operator at shapes whose
launches would leave the device half empty, against the oracle."""
import contextlib
import math
import random

import pytest
import torch

import flag_attn
from flagattention_amd import _abi, _lib, flash
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


def test_native_rules_equal_the_python_ones():
    native, lib, rng = _lib.native(), _lib.get(), random.Random(13)
    dealt = 0
    for _ in range(1500):
        size = lambda top: int(top ** rng.random())   # noqa: E731
        B, H, M, N, D = size(20), size(70), size(40000), size(40000), rng.choice([16, 32, 64, 128])
        for causal in (False, True):
            args = (B, H, M, N, D, causal, rng.choice([1, 1, 4]), rng.random() < 0.5, rng.choice([256, 304]))
            kv, q = flash.gradient_pieces(*args)
            assert native.gradient_pieces(*args) == (kv, q), args
            assert 1 <= kv <= 16 and 1 <= q <= 16 and (kv == 1 or -(-M // 64) >= 8 * kv) and (q == 1 or -(-N // 64) >= 8 * q)
            dealt += kv > 1 or q > 1
        # a kept mask takes no more memory than q, k, v and o (equal heads and lengths), up to the rounding of 64 keys
        if native.keeps_mask(N, D):
            assert lib.fa_dropout_keep_words(32 * M, N) * 4 <= 32 * M * (4 * 2 * D + 8)
        else:
            assert lib.fa_dropout_keep_words(32 * M, N) * 4 > 32 * M * 4 * 2 * D
    assert dealt > 300


# a result, or a launch, per head group in turns or all in one; dS kept or formed again; slices or, without memory, none
@pytest.mark.parametrize("H,Hk,chunk", [(2, 2, 1), (4, 2, 1), (4, 2, 2)])
@pytest.mark.parametrize("D,heads", [(64, 0), (128, 2), (128, 8)])
@pytest.mark.parametrize("memory", [True, False])
def test_python_backward_in_pieces_on_the_simulator(monkeypatch, H, Hk, chunk, D, heads, memory):
    lib = simlib.get()
    monkeypatch.setattr(_lib, "get", lambda: lib)
    monkeypatch.setattr(torch.cuda, "device", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(flash, "ds_heads_per_launch", lambda *a, **k: min(heads, 2 * H))
    monkeypatch.setattr(flash, "dkdv_heads_per_slice", lambda *a: chunk)
    gen = torch.Generator().manual_seed(9)
    q, k, v, do = (torch.randn(2, h, t, D, generator=gen).bfloat16() for h, t in ((H, 90), (Hk, 140), (Hk, 140), (H, 90)))
    leaves, grads, scratch = [t.requires_grad_() for t in (q, k, v)], [], flash._scratch
    for pieces in ((1, 1), (1 if chunk > 1 else 2, 3)):
        monkeypatch.setattr(flash, "gradient_pieces", lambda *a: pieces)
        if pieces != (1, 1) and not memory:
            monkeypatch.setattr(flash, "_scratch", lambda shape, dtype, device: None if dtype == torch.float32 else scratch(shape, dtype, device))
        o = flash.FlashAttention.apply(*leaves, True, None, 0.0, False, False, False)
        grads.append(torch.autograd.grad(o, leaves, do))
    for name, whole, parts in zip(("dq", "dk", "dv"), *grads):   # each fp32 sum in another order, rounded once to bf16
        assert (whole.float() - parts.float()).abs().max() <= 2 ** -7 * whole.float().abs().max(), name


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Hk,M,N,D,causal,limit_mib", [
    (1, 4, 4, 2000, 2000, 64, True, 4096),
    (1, 2, 2, 1100, 3001, 128, True, 4096),
    (1, 8, 2, 1111, 1500, 128, False, 4096),
    (2, 2, 2, 2000, 2100, 128, True, 9),         # dS of one head at a time
    (3, 2, 1, 700, 2000, 16, False, 4096),
])
def test_native_backward_deals_as_the_python_one(monkeypatch, B, H, Hk, M, N, D, causal, limit_mib):
    monkeypatch.setattr(flash, "DS_WORKSPACE_LIMIT_MIB", limit_mib)
    gen = torch.Generator(device="cuda").manual_seed(6)
    q, k, v, do = (torch.randn(B, h, t, D, device="cuda", generator=gen).bfloat16() for h, t in ((H, M), (Hk, N), (Hk, N), (H, M)))
    leaves = [t.requires_grad_() for t in (q, k, v)]
    heads = flash.ds_heads_per_launch(_lib.get(), B, H, H // Hk, M, N, D)
    assert max(flash.gradient_pieces(B, H, M, N, D, causal, 1, heads > 0, 256)) > 1
    if limit_mib < 4096:
        assert 0 < heads < B * H
    python = flash.FlashAttention.apply(*leaves, causal, None, 0.0, False, False, False)
    for a, b in zip(torch.autograd.grad(flag_attn.flash_attention(*leaves, causal), leaves, do), torch.autograd.grad(python, leaves, do)):
        assert torch.equal(a, b)
