"""Launches of more workgroups than compute units under the causal mask deal their tiles by ``tile_of_workgroup``: every
tile exactly once for every grid, whatever the heads, the rounds and the remainders."""
import pytest
import torch

import flag_attn
from oracle import flash_attention, within_two_x

pytestmark = pytest.mark.gpu


# workgroups of 128 rows: just past one per compute unit, a second round that is not full and not a multiple of 8, a
# full one, an odd head count over several rounds, one head group per XCD over many rounds
@pytest.mark.parametrize("B,H,T,D", [(1, 257, 100, 32), (1, 97, 400, 64), (1, 131, 384, 16), (2, 64, 512, 64), (1, 129, 520, 64),
                                     (3, 43, 1030, 64), (1, 64, 2050, 32), (2, 45, 640, 128)])
def test_every_tile_is_dealt_once(B, H, T, D):
    gen = torch.Generator(device="cuda").manual_seed(B * 1000 + H)
    q, k, v = (torch.randn(B, H, T, D, device="cuda", dtype=torch.bfloat16, generator=gen).requires_grad_() for _ in range(3))
    do = torch.randn(B, H, T, D, device="cuda", dtype=torch.bfloat16, generator=gen)

    def run(attention, **kw):
        o, _, total = attention(q, k, v, True, return_log_normalizer=True, return_total_attention=True, **kw)[:3]
        return (o, total) + torch.autograd.grad(o, (q, k, v), do)
    got = run(flag_attn.flash_attention)
    same, ref = (run(flash_attention, upcast=u) for u in (False, True))
    for name, h, s, r in zip(("o", "total", "dq", "dk", "dv"), got, same, ref):
        ok, e_h, e_s = within_two_x(h, s, r)
        assert ok, f"{name}: {e_h:.3e} against {e_s:.3e} of torch at the same precision"
