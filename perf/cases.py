"""The work that programs have the attention operators do, as cases that can be timed one by one.

A case is a dict of plain values.  ``op`` names the entry point:

* ``flash``     ``flash_attention``: training steps (``grad``), prefill, prefill chunks, dense decode;
* ``piecewise`` ``piecewise_attention``, forward and backward;
* ``paged``     ``paged_attention``, one token per sequence over a block-table-indexed cache.

``listed()`` holds one case for each kind of use, ``draw()`` gives further ones of the same ranges.
"""
import random

import torch

import flag_attn

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _flash(B, Hq, Hk, M, N, D, dtype, causal, grad=False, layout="BHTD", dropout=0.0, scores=False):
    """``layout`` is the order in which q, k, v (and so o and its gradient) lie in memory; ``scores`` asks for the
    log-normalizer and the column sums of the attention matrix as well."""
    return {"op": "flash", "B": B, "Hq": Hq, "Hk": Hk, "M": M, "N": N, "D": D, "dtype": dtype, "causal": causal,
            "grad": grad, "layout": layout, "dropout": dropout, "scores": scores}


def _piecewise(B, H, T, D, w, dtype, causal, layout="BHTD"):
    return {"op": "piecewise", "B": B, "H": H, "T": T, "D": D, "w": w, "dtype": dtype, "causal": causal,
            "layout": layout}


def _paged(seqs, Hq, Hkv, D, block, ctx_min, ctx_max, dtype):
    return {"op": "paged", "seqs": seqs, "Hq": Hq, "Hkv": Hkv, "D": D, "block": block, "ctx_min": ctx_min,
            "ctx_max": ctx_max, "dtype": dtype}


def listed():
    return [
        # one request that generates: a token against a short dense cache, grouped heads; all latency
        dict(_flash(1, 32, 8, 1, 1024, 128, "fp16", True), name="decode one request 1k"),
        # a handful of requests in a serving loop, short and uneven contexts; all latency
        dict(_paged(4, 32, 8, 128, 16, 100, 2000, "bf16"), name="paged 4 seqs to 2k"),
        # a serving batch with contexts of every length between 512 and 8192
        dict(_paged(64, 32, 8, 128, 16, 512, 8192, "fp16"), name="paged 64 seqs to 8k"),
        # long-context decode of a small batch over a dense cache
        dict(_flash(4, 32, 8, 1, 32768, 128, "fp16", True), name="decode batch 4 32k"),
        # an encoder layer on a short batch, forward and backward: launches and host work
        dict(_flash(2, 4, 4, 512, 512, 64, "fp16", False, grad=True), name="train small encoder"),
        # a training step of ordinary size
        dict(_flash(4, 16, 16, 2048, 2048, 128, "bf16", True, grad=True), name="train 2k"),
        # a training step on a long sequence
        dict(_flash(1, 32, 32, 8192, 8192, 128, "bf16", True, grad=True), name="train 8k"),
        # the longest sequence of the benchmark sweeps
        dict(_flash(1, 16, 16, 32768, 32768, 128, "bf16", True, grad=True), name="train 32k"),
        # head size 64, grouped heads, a length no tile divides, tokens before heads in memory
        dict(_flash(2, 32, 8, 4001, 4001, 64, "fp16", True, grad=True, layout="BTHD"), name="train d64 gqa ragged"),
        # a chunk of a prompt against the keys so far, with the scores that a cache-eviction policy reads
        dict(_flash(1, 32, 8, 1000, 8200, 128, "bf16", True, layout="BTHD", scores=True), name="prefill chunk scores"),
        # two score functions by distance, forward and backward
        dict(_piecewise(2, 32, 4096, 128, 1024, "bf16", True), name="piecewise train 4k"),
        # a training step with dropout
        dict(_flash(4, 16, 16, 1024, 1024, 64, "bf16", True, grad=True, dropout=0.1), name="train 1k dropout"),
    ]


def _between(rng, lo, hi):
    """A whole number of lo .. hi, its logarithm evenly spread."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _heads(rng, D):
    """(query heads, key/value heads) around 2048 / D query heads."""
    hq = rng.choice([4, 8, 16, 32]) if D >= 128 else rng.choice([4, 8, 16, 32, 64])
    return hq, hq // rng.choice([g for g in (1, 1, 1, 2, 4, 8) if hq % g == 0])


def draw(rng: random.Random):
    kind = rng.choice(["train"] * 6 + ["prefill"] * 3 + ["decode"] * 3 + ["paged"] * 4 + ["piecewise"] * 2 + ["dropout"] * 2)
    dtype, layout = rng.choice(["bf16", "bf16", "fp16"]), rng.choice(["BHTD", "BTHD"])
    if kind == "train":
        D = rng.choice([128, 128, 128, 64, 64, 32])
        hq, hk = _heads(rng, D)
        T = _between(rng, 300, 24000)
        N = T if rng.random() < 0.8 else T + rng.randrange(1, 500)
        B = max(1, min(8, 32768 // T, int(rng.choice([1, 2, 4, 8]))))
        return _flash(B, hq, hk, T, N, D, dtype, rng.random() < 0.7, grad=True, layout=layout) if T * N * hq * B < 2 ** 33 \
            else _flash(1, 8, 8 // (hq // hk), T, N, D, dtype, True, grad=True, layout=layout)
    if kind == "prefill":
        D = rng.choice([128, 128, 64])
        hq, hk = _heads(rng, D)
        N = _between(rng, 500, 32000)
        M = N if rng.random() < 0.4 else _between(rng, 64, min(N, 2048))
        B = 1 if N > 8000 else rng.choice([1, 2, 4])
        return _flash(B, hq, hk, M, N, D, dtype, True, layout=layout, scores=rng.random() < 0.3)
    if kind == "decode":
        D = rng.choice([128, 128, 64])
        hq, hk = _heads(rng, D)
        N, B = _between(rng, 500, 130000), _between(rng, 1, 64)
        B = max(1, min(B, 300000 // N))
        return _flash(B, hq, hk, rng.choice([1, 1, 1, 4]), N, D, dtype, True, layout=layout)
    if kind == "paged":
        D = rng.choice([128, 128, 128, 64, 256])
        hkv = rng.choice([2, 4, 8, 16])
        seqs, top = _between(rng, 1, 256), _between(rng, 200, 16000)
        seqs = max(1, min(seqs, 400000 * 8 // (top * hkv)))
        low = top if rng.random() < 0.3 else max(1, int(top * rng.random()))
        return _paged(seqs, hkv * rng.choice([1, 4, 8]), hkv, D, rng.choice([16, 16, 32]), low, top, dtype)
    if kind == "piecewise":
        D, H = rng.choice([128, 128, 64]), rng.choice([8, 16, 32])
        T = _between(rng, 400, 9000)
        return _piecewise(max(1, min(4, 8192 // T)), H, T, D, rng.randrange(T // 8, T), dtype, rng.random() < 0.8, layout)
    D = rng.choice([128, 64, 64])
    T, H = _between(rng, 256, 4000), rng.choice([8, 16])
    return _flash(max(1, min(4, 4096 // T)), H, H, T, T, D, dtype, rng.random() < 0.7, grad=True, layout=layout,
                  dropout=rng.choice([0.1, 0.2]))


class _Source:
    """Standard-normal tensors on the GPU, made from one seed."""

    def __init__(self, case, seed):
        self.dtype, self.layout = _DTYPES[case["dtype"]], case.get("layout", "BHTD")
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def __call__(self, B, H, T, D, grad=False):
        order = (B, H, T, D) if self.layout == "BHTD" else (B, T, H, D)
        t = torch.empty(order, dtype=self.dtype, device="cuda").normal_(0.0, 1.0, generator=self.gen)
        return (t if self.layout == "BHTD" else t.transpose(1, 2)).requires_grad_(grad)


def _context_lens(case):
    """The lengths of a paged batch, evenly spread from the shortest to the longest."""
    n, lo, hi = case["seqs"], case["ctx_min"], case["ctx_max"]
    return [hi - (hi - lo) * i // max(1, n - 1) for i in range(n)]


def prepare(case, seed):
    normal = _Source(case, seed)
    if case["op"] == "flash":
        B, Hq, Hk, M, N, D, grad = (case[n] for n in ("B", "Hq", "Hk", "M", "N", "D", "grad"))
        q, k, v = normal(B, Hq, M, D, grad), normal(B, Hk, N, D, grad), normal(B, Hk, N, D, grad)
        if case["dropout"] > 0:
            torch.cuda.manual_seed(seed)    # the mask is drawn from the device's default generator
        return {"case": case, "q": q, "k": k, "v": v, "do": normal(B, Hq, M, D) if grad else None}
    if case["op"] == "piecewise":
        shape = (case["B"], case["H"], case["T"], case["D"])
        return {"case": case, "in": [normal(*shape, grad=True) for _ in range(5)], "do": normal(*shape)}
    rng = random.Random(seed)
    lens, block = _context_lens(case), case["block"]
    rng.shuffle(lens)
    widest = -(-case["ctx_max"] // block)
    blocks = sum(-(-n // block) for n in lens) + 16     # a pool with a few blocks free
    free = torch.randperm(blocks, generator=torch.Generator().manual_seed(seed)).tolist()
    tables = torch.zeros((len(lens), widest), dtype=torch.int32)
    for i, n in enumerate(lens):
        own = -(-n // block)
        tables[i, :own] = torch.tensor(free[:own], dtype=torch.int32)
        del free[:own]
    return {"case": case, "q": normal(1, len(lens), case["Hq"], case["D"])[0],
            "kc": normal(blocks, case["Hkv"], block, case["D"]), "vc": normal(blocks, case["Hkv"], block, case["D"]),
            "lens": torch.tensor(lens, dtype=torch.int32, device="cuda"), "tables": tables.cuda(), "longest": max(lens),
            "scale": case["D"] ** -0.5}


def run(state):
    case = state["case"]
    if case["op"] == "paged":
        return flag_attn.paged_attention(state["q"], state["kc"], state["vc"], state["lens"], state["tables"],
                                         state["scale"], state["longest"])
    if case["op"] == "piecewise":
        o = flag_attn.piecewise_attention(*state["in"], case["w"], causal=case["causal"])
        return (o.detach(),) + torch.autograd.grad(o, state["in"], state["do"])
    q, k, v = state["q"], state["k"], state["v"]
    if case["scores"]:
        return flag_attn.flash_attention(q, k, v, causal=case["causal"], return_log_normalizer=True,
                                         return_total_attention=True)[:3]
    o = flag_attn.flash_attention(q, k, v, causal=case["causal"], dropout_p=case["dropout"])
    if not case["grad"]:
        return o
    return (o.detach(),) + torch.autograd.grad(o, (q, k, v), state["do"])


def _pairs(M, N, causal):
    """Unmasked (query, key) pairs; the causal mask is aligned at the last query and key."""
    if not causal:
        return M * N
    first = max(0, M - N)       # rows before this one see no key
    n = M - first
    return n * (N - M + first + 1) + n * (n - 1) // 2


def work(case):
    """A product is two operations per pair and channel: two products forward, five backward, one for the column sums;
    each score is one dot product in piecewise attention too."""
    D = case["D"]
    if case["op"] == "paged":
        rows, tokens = case["seqs"] * case["Hq"], sum(_context_lens(case))
        tables = 4 * sum(-(-n // case["block"]) for n in _context_lens(case))
        return {"bytes": 2 * 2 * tokens * case["Hkv"] * D + 2 * 2 * rows * D + tables + 4 * case["seqs"],
                "flops": 4 * tokens * case["Hq"] * D}
    if case["op"] == "piecewise":
        rows = case["B"] * case["H"] * case["T"]
        # q1, k1, q2, k2, v, o forward; those, the gradient of o and five gradients backward
        return {"bytes": 2 * rows * D * (6 + 6 + 1 + 5), "flops": 14 * case["B"] * case["H"] * D * _pairs(case["T"], case["T"], case["causal"])}
    q, k = case["B"] * case["Hq"] * case["M"] * D, case["B"] * case["Hk"] * case["N"] * D
    product = 2 * case["B"] * case["Hq"] * D * _pairs(case["M"], case["N"], case["causal"])
    size, flops = 2 * (2 * q + 2 * k), 2 * product      # q, k, v, o
    if case["grad"]:
        size, flops = size + 2 * (4 * q + 4 * k), flops + 5 * product    # q, k, v, o, do; dq, dk, dv
    if case["scores"]:
        size, flops = size + 4 * case["B"] * case["Hq"] * (case["M"] + case["N"]), flops + product
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """Probabilities and score gradients are rounded to the input type between the products: a few units of its last
    place (2^-8 for bf16, 2^-11 for fp16) in the 2-norm."""
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}
