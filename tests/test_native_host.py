"""The native host path of the operators (``csrc/host.cpp``) against the Python form of the same host logic:
the launch decisions number by number (no GPU needed), and on the GPU the results bit for bit."""
import random

import pytest
import torch

import flag_attn
from flagattention_amd import _lib, flash, paged, piecewise, split_kv


def test_native_decisions_equal_the_python_ones():
    native, lib, rng = _lib.native(), _lib.get(), random.Random(7)
    shapes = [(1, 1, 1, 1, 1, 16), (4, 32, 8, 1, 32768, 128), (1, 32, 32, 1024, 8192, 128), (1, 16, 16, 32768, 32768, 128),
              (1, 8, 8, 1024, 1024, 128), (1, 8, 8, 1024, 1023, 128), (1, 32, 8, 256, 1024, 128), (1, 32, 8, 255, 4096, 128)]
    for _ in range(400):
        Hk, size = rng.choice([1, 2, 4, 8, 16]), lambda top: int(top ** rng.random())
        shapes.append((size(200), Hk * rng.choice([1, 2, 3, 4, 8]), Hk, size(20000), size(200000), rng.choice([16, 32, 64, 128])))
    for B, H, Hk, M, N, D in shapes:
        for cus, limit in ((256, 4096), (304, 700)):
            got = native.decisions(B, H, Hk, M, N, D, cus, limit)
            chosen = split_kv.choose_num_splits(B, H, Hk, M, N, cus, 2)
            flash_limit, flash.DS_WORKSPACE_LIMIT_MIB = flash.DS_WORKSPACE_LIMIT_MIB, limit
            try:
                heads = [flash.ds_heads_per_launch(lib, B, H, g, M, N, D, grids=n) for g, n in ((H // Hk, 1), (1, 2))]
            finally:
                flash.DS_WORKSPACE_LIMIT_MIB = flash_limit
            want = {"num_splits_heuristic": split_kv.num_splits_heuristic(B, H, M, N, 16, 128, cus, 128),
                    "choose_num_splits": chosen, "split_size": split_kv._split_size(N, chosen),
                    "wide_key_splits": flash.wide_key_splits(B, H, M, N, D, cus),
                    "dkdv_heads_per_slice": flash.dkdv_heads_per_slice(B, H, H // Hk, N, cus),
                    "ds_heads_per_launch": heads[0], "ds_heads_per_launch_piecewise": heads[1],
                    "balanced_workgroups": paged.choose_launch(B, Hk, H // Hk, D, N, cus)[1]}
            assert got == want, (B, H, Hk, M, N, D, cus, limit)


def randn(*shape, dtype=torch.bfloat16, layout="BHTD", grad=False):
    B, H, T, D = shape
    t = torch.randn(*shape, dtype=dtype, device="cuda") if layout == "BHTD" else \
        torch.randn(B, T, H, D, dtype=dtype, device="cuda").transpose(1, 2)
    return t.requires_grad_(grad)


def same(a, b):
    layout = [[s for n, s in zip(t.shape, t.stride()) if n > 1] for t in (a, b)]
    return torch.equal(a, b) and layout[0] == layout[1] and a.dtype == b.dtype and a.requires_grad == b.requires_grad


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Hk,M,N,D,causal,layout", [
    (1, 32, 8, 1, 1024, 128, True, "BHTD"),       # split decode; gradients of a group added
    (1, 8, 8, 1, 1030, 64, False, "BTHD"),        # decode in one piece: no merge
    (1, 32, 8, 300, 5000, 128, True, "BTHD"),     # pieces of the key axis through the 256-row kernel
    (2, 4, 4, 513, 511, 64, False, "BHTD"),       # dense; recomputing backward
    (1, 8, 2, 1025, 1030, 128, True, "BTHD"),     # dS kept, gradients of a group added
])
def test_native_flash_equals_the_python_path(B, H, Hk, M, N, D, causal, layout):
    q, k, v = (randn(B, h, t, D, layout=layout, grad=True) for h, t in ((H, M), (Hk, N), (Hk, N)))
    do = randn(B, H, M, D)
    native = flag_attn.flash_attention(q, k, v, causal, None, 0.0, True, True)
    python = flash.FlashAttention.apply(q, k, v, causal, None, 0.0, True, True, False)
    for a, b in zip(native[:3], python[:3]):
        assert same(a, b)
    assert native[3:] == (None, None)
    # (bound for fp32 sums in another order and one rounding to bf16; test_gradient_pieces.py holds both to the same order)
    for a, b in zip(torch.autograd.grad(native[0], (q, k, v), do), torch.autograd.grad(python[0], (q, k, v), do)):
        assert a.shape == b.shape and a.dtype == b.dtype
        assert (a.float() - b.float()).abs().max() <= 2 ** -7 * b.float().abs().max()
    with torch.no_grad():
        assert torch.equal(flag_attn.flash_attention(q, k, v, causal), native[0])


@pytest.mark.gpu
def test_native_dropout_draws_like_the_python_path():
    q, k, v = (randn(8, 16, 200, 64, dtype=torch.float16, grad=True) for _ in range(3))
    outs = []
    for call in (flag_attn.flash_attention, flash.FlashAttention.apply):
        torch.cuda.manual_seed(-5)
        for _ in range(2):   # the second call finds the generator advanced
            outs.append(call(q, k, v, True, None, 0.2, False, False, True))
    assert outs[0][3:] == outs[2][3:] and outs[1][3:] == outs[3][3:] and outs[0][4] != outs[1][4]
    assert torch.equal(outs[0][0], outs[2][0]) and torch.equal(outs[1][0], outs[3][0])


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Hk,M,N,D,causal", [
    (8, 16, 16, 129, 129, 64, True),       # rows and keys one past a tile
    (8, 16, 8, 31, 97, 16, False),         # less than a block of rows, three blocks of keys
    (4, 32, 32, 160, 33, 32, True),        # rows that see no key
    (16, 16, 16, 100, 64, 128, False),
    (4, 16, 4, 1100, 1030, 128, True),     # dS kept
])
def test_kept_dropout_mask_gives_the_gradients_of_a_drawn_one(B, H, Hk, M, N, D, causal):
    """The native path hands the forward's mask to the backward as bits, the Python path draws it again: the same
    elements survive, so all results are equal bit for bit -- with a counter whose upper word changes inside the call."""
    q, k, v = (randn(B, h, t, D, grad=True) for h, t in ((H, M), (Hk, N), (Hk, N)))
    do = randn(B, H, M, D)
    gen = torch.cuda.default_generators[0]
    results = []
    for call in (flag_attn.flash_attention, flash.FlashAttention.apply):
        gen.manual_seed(2 ** 40 + 3)
        gen.set_offset(2 ** 32 - 4 * (B * H * M * N // 8))
        o, _, _, seed, offset = call(q, k, v, causal, None, 0.3, False, False, True)
        assert offset < 2 ** 32 < offset + B * H * M * N
        results.append((o,) + torch.autograd.grad(o, (q, k, v), do))
    for name, a, b in zip(("o", "dq", "dk", "dv"), *results):
        assert torch.equal(a, b), name


@pytest.mark.gpu
def test_calls_the_native_path_does_not_take_still_raise():
    q, k = randn(1, 4, 64, 64), randn(1, 3, 64, 64)
    with pytest.raises(AssertionError):
        flag_attn.flash_attention(q, k, k)
    with pytest.raises(AssertionError):
        flag_attn.flash_attention(q, q, q, dropout_p=1.5)
    with pytest.raises(AssertionError):
        flag_attn.flash_attention(q.float(), q.float(), q.float())


@pytest.mark.gpu
@pytest.mark.parametrize("T,D,w", [(1024, 128, 300), (257, 64, 100)])
def test_native_piecewise_equals_the_python_path(T, D, w):
    ins = [randn(1, 4, T, D, layout="BTHD", grad=True) for _ in range(5)]
    do = randn(1, 4, T, D)
    a = flag_attn.piecewise_attention(*ins, w, causal=True)
    b = piecewise.PiecewiseAttention.apply(*ins, w, True, None)
    assert same(a, b)
    for x, y in zip(torch.autograd.grad(a, ins, do), torch.autograd.grad(b, ins, do)):
        assert torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["flash", "piecewise"])
def test_transforms_and_tracers_see_a_python_function(op):
    """Forward-mode tangents, functorch transforms and the tracer meet the same function that they would without the native
    path: what torch refuses is refused, and a trace holds the call and not its results."""
    from torch.autograd import forward_ad
    if op == "flash":
        native, python = (lambda *t: flag_attn.flash_attention(*t[:3], True)), \
            (lambda *t: flash.FlashAttention.apply(*t[:3], True, None, 0.0, False, False, False))
    else:
        native, python = (lambda *t: flag_attn.piecewise_attention(*t, 40, True)), \
            (lambda *t: piecewise.PiecewiseAttention.apply(*t, 40, True, None))
    ins, others = ([randn(1, 2, 96, 64) for _ in range(5)] for _ in range(2))

    def tangents(f):
        with forward_ad.dual_level():
            return f(*[forward_ad.make_dual(t, torch.ones_like(t)) for t in ins])

    def outcome(f):
        try:
            return f()
        except Exception as e:   # noqa: BLE001 - compared below
            return type(e)
    for form in (tangents, lambda f: torch.func.grad(lambda q: f(q, *ins[1:]).sum())(ins[0]),
                 lambda f: torch.vmap(lambda q: f(q, *ins[1:]))(torch.stack([ins[0]] * 2)),
                 lambda f: torch.jit.trace(f, tuple(ins), check_trace=False)(*others)):
        a, b = outcome(lambda: form(native)), outcome(lambda: form(python))
        assert isinstance(a, torch.Tensor) == isinstance(b, torch.Tensor), (a, b)
        assert torch.equal(a, b) if isinstance(a, torch.Tensor) else a is b, (a, b)


def paged_arguments():
    lens, table = torch.tensor([40, 9], dtype=torch.int32, device="cuda"), torch.arange(6, device="cuda").reshape(2, 3)
    return randn(1, 2, 4, 64)[0], randn(6, 4, 16, 64), randn(6, 4, 16, 64), lens, table


@pytest.mark.gpu
def test_paged_call_is_made_in_python_where_something_listens():
    """As for the other operators: the native path launches past the dispatcher, so it takes no call that a dispatch mode, a
    tracer, a transform or a tangent should see."""
    from torch.autograd import forward_ad
    from torch.utils._python_dispatch import TorchDispatchMode
    q, *rest = paged_arguments()

    def native(query):
        return _lib.native().paged(query, *rest, 0.125, 40)

    class Recorder(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    assert isinstance(native(q), torch.Tensor)
    seen, answers = [], []
    with Recorder():
        flag_attn.paged_attention(q, *rest, 0.125, 40)
    assert any("empty" in name for name in seen)
    with forward_ad.dual_level():
        answers.append(native(forward_ad.make_dual(q, torch.ones_like(q))))
    torch.vmap(lambda query: answers.append(native(query)) or query)(torch.stack([q, q]))
    torch.jit.trace(lambda query: answers.append(native(query)) or query, (q,), check_trace=False)
    assert len(answers) == 3 and all(a is NotImplemented for a in answers)


@pytest.mark.gpu
def test_tensor_subclasses_get_their_own_type_back():
    """A subclass without __torch_dispatch__ is what the Python form's torch.empty_like makes of it; parameters are taken as
    the tensors they are."""
    class Named(torch.Tensor):
        pass

    q, k, v, q2, k2 = (randn(1, 4, 96, 64) for _ in range(5))
    query, *rest = paged_arguments()
    for kind in (Named, torch.nn.Parameter):
        own = (lambda t: t.as_subclass(Named)) if kind is Named else torch.nn.Parameter
        outs = [flag_attn.flash_attention(own(q), k, v), flag_attn.piecewise_attention(own(q), k, q2, k2, v, 40),
                flag_attn.paged_attention(own(query), *rest, 0.125, 40)]
        assert [type(o) for o in outs] == [Named if kind is Named else torch.Tensor] * 3
        assert [o.requires_grad for o in outs] == [kind is not Named] * 2 + [False]
    plain = flag_attn.flash_attention(q, k, v), flag_attn.piecewise_attention(q, k, q2, k2, v, 40), flag_attn.paged_attention(query, *rest, 0.125, 40)
    for a, b in zip(outs, plain):
        assert torch.equal(a, b)
