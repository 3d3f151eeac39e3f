"""NaN and infinities in the inputs reach the output by every route: the whole key axis in one workgroup, pieces of it merged
afterwards (every merge variant), the decode kernel and the three forms of the paged one.  A row is NaN exactly where
the oracle's is; a row without keys stays zero with a log-normalizer of -inf."""
import math

import pytest
import torch

import flag_attn
from flagattention_amd import _abi, _lib, split_kv
from oracle import flash_attention, paged_attention
from tests.sim import simlib

NAN, INF = float("nan"), float("inf")
POISONS = [("q", NAN), ("q", INF), ("k", NAN), ("k", INF), ("k", -INF), ("v", NAN), ("v", INF)]


@pytest.fixture(params=["simulator", pytest.param("gpu", marks=pytest.mark.gpu)])
def target(request):
    return (simlib.get(), "cpu") if request.param == "simulator" else (_lib.get(), "cuda")


def same_special_values(out, ref, lse=None, ref_lse=None):
    """Sums of at most 500 products of 16-bit values of order 1: 2e-2 covers the rounding of the results and of P."""
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    assert torch.equal(out.isposinf(), ref.isposinf()) and torch.equal(out.isneginf(), ref.isneginf())
    assert ((out.float() - ref.float())[torch.isfinite(ref)].abs() < 2e-2).all()
    if lse is not None:   # torch.logsumexp of a row with a score of +inf is +inf, the kernels give NaN
        assert torch.equal(lse.isneginf(), ref_lse.isneginf())
        assert torch.equal(torch.isfinite(lse), torch.isfinite(ref_lse))


def poisoned(tensors, what, value, row):
    tensors = {n: t.clone() for n, t in tensors.items()}
    tensors[what][..., row if what != "q" else 7, 5] = value
    return tensors


def dense_routes(lib, q, k, v, causal):
    """(name, o, lse) by every forward kernel and merge."""
    (B, H, M, D), N, scale = q.shape, k.shape[2], q.shape[-1] ** -0.5

    def results():
        return torch.full_like(q, 7.0), torch.full((B, H, M), 7.0, device=q.device)
    for block_m in (128, 256):
        if block_m == 128 or (D == 128 and M >= 256):
            o, lse = results()
            _abi.fa_fwd(lib, q, k, v, o, lse, causal, scale, block_m=block_m)
            yield f"whole, {block_m} rows", o, lse
    for pieces in (2, 7, 16):   # up to 4, up to 8 and more pieces: three kernels
        o, lse = results()
        _abi.fa_fwd_pieces(lib, q, k, v, o, lse, causal, scale, pieces)
        yield f"{pieces} pieces", o, lse
    for splits in (1, 2, 4):    # the decode kernel, or 256-row workgroups; partial results in fp16
        if split_kv._split_size(N, splits) * (splits - 1) >= N:
            continue
        o, lse = results()
        part_o = torch.full((B, H, splits, M, D), 7.0, dtype=torch.float16, device=q.device)
        part_lse = torch.full((B, H, splits, M), 7.0, device=q.device)
        _abi.fa_splitkv_fwd(lib, q, k, v, part_o, part_lse, causal, scale, splits, split_kv._split_size(N, splits))
        _abi.fa_splitkv_combine(lib, part_o, part_lse, o, lse, splits)
        yield f"{splits} splits", o, lse


@pytest.mark.parametrize("what,value", POISONS)
@pytest.mark.parametrize("M,N,D,causal,dtype", [(40, 400, 64, False, torch.float16), (40, 400, 128, True, torch.bfloat16),
                                                 (70, 40, 16, True, torch.float16), (257, 129, 128, True, torch.float16)])
def test_dense(target, what, value, M, N, D, causal, dtype):
    if what == "v" and causal:   # p v with p = 0 is NaN in the oracle and in tiles that hold a hidden key, not in others
        causal = False
    lib, device = target
    gen = torch.Generator().manual_seed(4)
    t = {n: torch.randn(1, 1, rows, D, generator=gen).to(dtype) for n, rows in (("q", M), ("k", N), ("v", N))}
    t = poisoned(t, what, value, N - 15)
    ref, ref_lse, _ = flash_attention(*t.values(), causal, upcast=True, return_log_normalizer=True)
    q, k, v = (x.to(device) for x in t.values())
    for name, o, lse in dense_routes(lib, q, k, v, causal):
        print(name, flush=True)
        same_special_values(o.cpu(), ref, lse.cpu(), ref_lse)


@pytest.mark.parametrize("what,value", POISONS[::2])
@pytest.mark.parametrize("G,D,dtype", [(2, 32, torch.bfloat16), (1, 64, torch.float16)])
def test_paged(target, what, value, G, D, dtype):
    lib, device = target
    gen = torch.Generator().manual_seed(5)
    lens, Hk, block, scale = torch.tensor([500, 37], dtype=torch.int32), 1, 16, D ** -0.5
    table = torch.randperm(80, generator=gen)[:64].reshape(2, 32)
    q = torch.randn(2, G, D, generator=gen).to(dtype)
    caches = {n: torch.randn(80, Hk, block, D, generator=gen).to(dtype) for n in "kv"}
    if what == "q":
        q[0, 0, 5] = value
    else:
        caches[what][table[0, 30], :, 3, 5] = value
    ref = paged_attention(q, caches["k"], caches["v"], table, lens, scale)
    q, kc, vc, lens, table = (x.to(device) for x in (q, caches["k"], caches["v"], lens, table))
    for parts in (1, 4):
        out, shape = torch.full_like(q, 7.0), (2, Hk, parts, G)
        part = [None] * 3 if parts == 1 else [torch.full(shape + (D,), 7.0, dtype=dtype, device=device)] + \
            [torch.full(shape, 7.0, device=device) for _ in range(2)]
        _abi.paged_attn(lib, out, q, kc, vc, lens, table, scale, 0 if parts == 1 else 128, parts, *part)
        if parts > 1:
            _abi.paged_reduce(lib, out, *part, lens, Hk, 128, parts)
        same_special_values(out.cpu(), ref)
    for wgs in (3, 12):   # ranges that cross pairs; a piece per workgroup, partials shared between the merge's threads
        out = torch.full_like(q, 7.0)
        ws = torch.full((lib.paged_attn_balanced_workspace(wgs, D) // 4,), 7.0, device=device)
        _abi.paged_attn_balanced(lib, out, q, kc, vc, lens, table, scale, ws, wgs)
        same_special_values(out.cpu(), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Hk,M,N,D", [
    (1, 32, 8, 1, 4000, 128),       # decode kernel and merge
    (1, 8, 8, 4, 600, 64),          # decode kernel, fewer keys
    (1, 32, 8, 100, 8200, 128),     # pieces of the 128-row kernel
    (1, 32, 32, 1024, 8192, 128),   # pieces of the 256-row kernel
    (8, 16, 16, 200, 300, 64),      # whole axis
])
@pytest.mark.parametrize("what", ["q", "k"])
def test_public_call(B, H, Hk, M, N, D, what):
    gen = torch.Generator(device="cuda").manual_seed(6)
    t = {n: torch.randn(B, h, rows, D, device="cuda", generator=gen).bfloat16() for n, h, rows in (("q", H, M), ("k", Hk, N), ("v", Hk, N))}
    row = 0 if what == "q" else N - M
    t[what][0, 0, row, 3] = NAN
    o, lse, total, *_ = flag_attn.flash_attention(*t.values(), causal=True, return_log_normalizer=True, return_total_attention=True)
    hit = torch.zeros(B, H, M, dtype=torch.bool, device="cuda")
    hit[0, :1 if what == "q" else H // Hk, :1 if what == "q" else None] = True    # the row itself, or all rows: they all see that key
    assert torch.equal(torch.isnan(o), hit[..., None].expand_as(o)) and torch.equal(torch.isnan(lse), hit)
    assert torch.isfinite(lse[~hit]).all() and torch.isnan(total[0, 0]).any() and torch.isfinite(total[0, -1]).all()


def test_dropped_key_still_counts():
    """A NaN score whose probability the dropout drops is part of the row sum."""
    lib, gen = simlib.get(), torch.Generator().manual_seed(8)
    q, k, v = (torch.randn(1, 1, rows, 64, generator=gen).half() for rows in (40, 100, 100))
    k[..., 50, 3] = NAN
    o, lse = torch.full_like(q, 7.0), torch.full((1, 1, 40), 7.0)
    _abi.fa_fwd(lib, q, k, v, o, lse, False, 1 / math.sqrt(64), dropout=(0.5, 3, 0))
    assert torch.isnan(o).all() and torch.isnan(lse).all()
