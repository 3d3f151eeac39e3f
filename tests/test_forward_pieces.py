"""The keys of a 128-row block dealt to several workgroups (``fa_fwd_pieces``): the rule, and the results over all ways in
which pieces, tiles and masks can end."""
import random

import pytest
import torch

import flag_attn
from flagattention_amd import _abi, _lib, flash
from oracle import flash_attention, within_two_x


def test_native_rule_equals_the_python_one():
    native, rng = _lib.native(), random.Random(11)
    for _ in range(600):
        Hk, size = rng.choice([1, 2, 4, 8, 16]), lambda top: int(top ** rng.random())
        shape = (size(60), Hk * rng.choice([1, 2, 4, 8]), Hk, size(5000), size(60000), rng.choice([16, 32, 64, 128]))
        for split in (False, True):
            n = flash.forward_pieces(*shape, split, 256)
            assert native.forward_pieces(*shape, split, 256) == n, shape
            rows, keys = -(-shape[3] // 128) * shape[0] * shape[1], -(-shape[4] // 64)
            assert n == 0 or (2 <= n <= 32 and n * rows <= 1024 and keys >= 3 * n)


def case(B, H, Hk, M, N, D, dtype, layout="BHTD"):
    gen = torch.Generator(device="cuda").manual_seed(M * 7 + N)
    def randn(h, t):
        x = torch.randn((B, h, t, D) if layout == "BHTD" else (B, t, h, D), device="cuda", dtype=dtype, generator=gen)
        return x if layout == "BHTD" else x.transpose(1, 2)
    return randn(H, M), randn(Hk, N), randn(Hk, N)


def compare(got, q, k, v, causal):
    same, ref = (flash_attention(q, k, v, causal, upcast=u, return_log_normalizer=True)[:2] for u in (False, True))
    for name, h, s, r in zip(("o", "lse"), got, same, ref):
        hidden = torch.isinf(r)
        assert torch.equal(torch.isinf(h), hidden)
        ok, e_h, e_s = within_two_x(h.masked_fill(hidden, 0), s.masked_fill(hidden, 0), r.masked_fill(hidden, 0))
        assert ok, f"{name}: {e_h:.3e} against {e_s:.3e} of torch at the same precision"


# pieces without a tile (more pieces than tiles, under the causal mask for the upper rows), one row, tails of both axes,
# rows that see no key, every merge variant (up to 4, up to 8, more pieces)
@pytest.mark.gpu
@pytest.mark.parametrize("pieces", [1, 2, 3, 7, 16, 64])
@pytest.mark.parametrize("M,N,causal", [(1, 65, True), (127, 1030, False), (129, 128, True), (300, 777, True), (257, 100, True)])
@pytest.mark.parametrize("D,dtype,layout", [(128, torch.bfloat16, "BHTD"), (64, torch.float16, "BTHD"), (32, torch.bfloat16, "BTHD"),
                                            (16, torch.float16, "BHTD")])
def test_pieces_against_the_oracle(pieces, M, N, causal, D, dtype, layout):
    q, k, v = case(2, 4, 2, M, N, D, dtype, layout)
    o, lse = torch.full_like(q, float("nan")), torch.full((2, 4, M), float("nan"), device="cuda")
    _abi.fa_fwd_pieces(_lib.get(), q, k, v, o, lse, causal, D ** -0.5, pieces)
    compare((o, lse), q, k, v, causal)


# calls that the rule takes here, from the whole-axis launch and from the decode kernel
@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Hk,M,N,D,causal", [(1, 16, 4, 100, 4100, 128, True), (1, 16, 16, 300, 3001, 64, True),
                                                  (1, 8, 8, 128, 8000, 128, False), (1, 8, 2, 1000, 1500, 32, True)])
def test_calls_in_pieces(B, H, Hk, M, N, D, causal):
    splits = flash.num_splits_heuristic(B, H, M, N, 16, 128, 256, 128)
    assert flash.forward_pieces(B, H, Hk, M, N, D, splits > 1, 256) > 1
    q, k, v = case(B, H, Hk, M, N, D, torch.bfloat16)
    native = flag_attn.flash_attention(q, k, v, causal, return_log_normalizer=True)[:2]
    compare(native, q, k, v, causal)
    python = flash.FlashAttention.apply(q, k, v, causal, None, 0.0, True, False, False)[:2]
    assert torch.equal(native[0], python[0]) and torch.equal(native[1], python[1])
