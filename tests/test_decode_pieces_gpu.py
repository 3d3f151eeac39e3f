"""Decode launches at the sizes where their pieces change: piece counts around the batches of the merge kernel, paged
batches of few pairs (one piece per workgroup) with lengths around a step and a unit of keys, and block sizes on both
sides of the rule that lets a load instruction take its block's address from scalar registers."""
import pytest
import torch

import flag_attn
from flagattention_amd import _abi, _lib, split_kv
from oracle import flash_attention as oracle_flash, paged_attention as oracle_paged, within_two_x

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [16, 64, 128])
@pytest.mark.parametrize("splits", [1, 2, 4, 5, 8, 9, 33, 70])
def test_split_and_merge(splits, D):
    """Any number of pieces gives the forward's result; the last piece ends inside a step, one row sees no key of it."""
    B, H, Hk, M, N = 1, 6, 2, 3, 128 * splits - 37
    lib, dtype = _lib.get(), torch.bfloat16
    q, k, v = (torch.randn(B, h, t, D, dtype=dtype, device="cuda") for h, t in ((H, M), (Hk, N), (Hk, N)))
    part_o = torch.full((B, H, splits, M, D), float("nan"), dtype=torch.float16, device="cuda")
    part_lse = torch.full((B, H, splits, M), float("nan"), device="cuda")
    o, lse = torch.full_like(q, float("nan")), torch.full((B, H, M), float("nan"), device="cuda")
    _abi.fa_splitkv_fwd(lib, q, k, v, part_o, part_lse, True, D ** -0.5, splits, split_kv._split_size(N, splits))
    _abi.fa_splitkv_combine(lib, part_o, part_lse, o, lse, splits)
    ref = oracle_flash(q, k, v, True, upcast=True, return_log_normalizer=True)
    same = oracle_flash(q, k, v, True, upcast=False, return_log_normalizer=True)
    for name, h, s, r in (("o", o, same[0], ref[0]), ("log-normalizer", lse, same[1], ref[1])):
        ok, e_hyp, e_same = within_two_x(h, s, r)
        assert ok, f"{name}: kernel err {e_hyp:.3e} vs same-precision torch err {e_same:.3e}"


@pytest.mark.parametrize("D,block", [(128, 16), (128, 12), (64, 16), (64, 4), (32, 16), (16, 16), (256, 32), (512, 16)])
@pytest.mark.parametrize("lens", [[1], [32, 33], [127, 0, 128, 129], [5000, 1, 700], list(range(100, 2200, 150))])
@pytest.mark.parametrize("group", [1, 5])
def test_paged_batches_of_few_pairs(lens, D, block, group):
    Hkv, n = 2, len(lens)
    widest = -(-max(lens) // block)
    q = torch.empty(n, Hkv * group, D, dtype=torch.float16, device="cuda").uniform_(-D ** -0.5, D ** -0.5)
    kc = torch.empty(n * widest, Hkv, block, D, dtype=torch.float16, device="cuda").uniform_(-D ** -0.5, D ** -0.5)
    vc = torch.empty_like(kc).uniform_(-D ** -0.5, D ** -0.5)
    table = torch.randperm(n * widest, device="cuda").view(n, widest)
    ctx = torch.tensor(lens, dtype=torch.int32, device="cuda")
    for s, length in enumerate(lens):   # what lies behind a sequence in its last block is not data
        if length % block:
            vc[table[s, length // block], :, length % block:] = float("nan")
    out = flag_attn.paged_attention(q, kc, vc, ctx, table.to(torch.int32), D ** -0.5, max(lens))
    ref = oracle_paged(q, kc, torch.nan_to_num(vc), table, ctx, D ** -0.5)
    assert torch.allclose(out, ref, atol=2e-3, rtol=1e-5)   # the reference's own bound for paged attention
