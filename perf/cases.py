"""The calls this framework is used for, as timed cases: SageAttention from 16-bit tensors (K mean, smoothing,
quantization, INT8 attention), SageAttention over a quantized K that is kept between calls, and the dense
flash_attention forward.

A case is a dict of plain values.  ``op`` names the sequence of public calls ``run`` makes:

* ``step``     per_block_int8(q, k, smooth_k=...) -> sage_attention(...): what a model's attention layer calls,
* ``sageattn`` the one-call wrapper, which can also return the natural-log log-sum-exp of the unsmoothed logits,
* ``kept``     sage_attention(...) on tensors that are quantized already: new queries against a K cache,
* ``flash``    flag_attn.flash_attention(...), the dense 16-bit forward.

Sizes are those of bench.py's workloads (c1 to c5), of the tests, or generic ones (grouped heads 32 / 8, a prompt of
odd length, a chunk of queries against a long cache, one query per sequence).
"""
import math

import torch

import flag_attn
from flag_attn import sage_attention as sa

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, op, b, h, hkv, m, n, d, dtype, layout="HND", causal=False, smooth=True, mask="none", out="same",
          lse=False, dropout=0.0, total=False, data="normal"):
    """``mask``: "none", or kind:type; kinds "padding" ([B, 1, 1, N], sequences of different lengths), "causal_padding"
    ([B, 1, M, N], both) and "bias" ([1, H, M, N], a position bias), type "bool" or the type of additive entries.
    ``data``: "normal", "offset" (K has a per-(head, channel) offset) or "outlier" (1 % of the (head, channel) pairs
    of Q and K scaled by 20, V uniform in (-1, 1)).  ``out``: output type ("same": that of the inputs)."""
    c = dict(op=op, b=b, h=h, hkv=hkv, m=m, n=n, d=d, dtype=dtype, layout=layout, causal=causal, smooth=smooth, mask=mask,
             out=out, lse=lse, dropout=dropout, total=total, data=data)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call, the reference's own unit-test shape: launches and host time are what counts
        _case("step_small", "step", 1, 2, 2, 256, 256, 64, "fp16"),
        # prefill of a batch of prompts
        _case("step_prefill", "step", 4, 32, 32, 4096, 4096, 128, "bf16"),
        # causal prefill, activations as the projections leave them ([B, N, H, D]), K with channel offsets
        _case("step_causal_nhd", "step", 2, 32, 32, 8192, 8192, 128, "bf16", layout="NHD", causal=True, data="offset"),
        # small heads with outlier channels, without smoothing
        _case("step_outlier_d64", "step", 8, 16, 16, 2048, 2048, 64, "fp16", smooth=False, data="outlier"),
        # attention of a diffusion transformer over one long sequence: the largest
        _case("step_long", "step", 1, 24, 24, 32768, 32768, 128, "bf16"),
        # the prefill of one prompt of odd length with grouped heads, through the one-call wrapper, with the log-sum-exp
        # (which partial results over several key ranges are merged by)
        _case("sageattn_odd_gqa_lse", "sageattn", 1, 32, 8, 3001, 3001, 128, "bf16", causal=True, lse=True),
        # a padded batch under the additive mask that model code builds: causal and padding in one, finite minimum
        _case("step_additive_mask", "step", 4, 16, 16, 1536, 1536, 128, "bf16", mask="causal_padding:bf16"),
        # chunked prefill: a chunk of new queries against a long quantized K
        _case("kept_chunk_gqa", "kept", 1, 32, 8, 512, 16384, 128, "fp16", causal=True, out="bf16"),
        # decoding: one new query per sequence, grouped heads, dense
        _case("flash_decode_gqa", "flash", 8, 32, 8, 1, 8192, 128, "bf16"),
        # dense causal prefill with grouped heads; the log normalizer is what a backward pass would keep
        _case("flash_causal_gqa", "flash", 2, 32, 8, 4096, 4096, 128, "bf16", causal=True, lse=True),
        # the forward pass of training with dropout
        _case("flash_dropout", "flash", 4, 16, 16, 2048, 2048, 64, "fp16", causal=True, dropout=0.1),
        # the attention every key receives (token pruning, cache eviction) beside the output
        _case("flash_total", "flash", 1, 16, 16, 4096, 4096, 128, "fp16", causal=True, lse=True, total=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi):
    """A sequence length, uniform over its logarithm: as it comes (odd ones among them) or a multiple of 64."""
    n = _log_int(rng, lo, hi)
    return n if rng.random() < 0.5 else max(64, n // 64 * 64)


# scores (batch x heads x queries x keys) of a drawn case at head_dim 128: half of the largest listed case, whose kernel
# is also the fastest per score; a third of that for the ops and options that cost more per score
_MAX_SCORES = 24 * 32768 * 32768 // 2


def draw(rng):
    op = rng.choice(["step", "step", "sageattn", "kept", "flash", "flash"])
    d = rng.choice([64, 128, 128])
    dtype = rng.choice(["fp16", "bf16"])
    h, hkv = rng.choice([(2, 2), (8, 8), (16, 16), (24, 24), (32, 32), (32, 8), (16, 2), (8, 1), (32, 4)])
    causal = rng.random() < 0.5
    mask, dropout, total, lse, layout, smooth, out = "none", 0.0, False, rng.random() < 0.3, "HND", True, "same"
    most, b_most = _MAX_SCORES, 8
    lo, hi = 64, 32768
    if op == "step":
        layout = rng.choice(["HND", "NHD"])
        smooth = rng.random() < 0.75
        if rng.random() < 0.4:
            mask = rng.choice(["padding", "causal_padding", "bias"]) + ":" + rng.choice(["bool", dtype, dtype, "fp32"])
            hi, most, b_most = 4096, _MAX_SCORES // 6, 4
            if mask.startswith("causal_padding"):
                causal = False  # (that mask holds the causal one already)
            if mask == "bias:bool":
                mask = "padding:bool"
        m = n = _length(rng, lo, hi)
        if not causal and mask == "none" and rng.random() < 0.25:
            n = _length(rng, 64, 4096)  # cross attention
    elif op == "sageattn":
        m = n = _length(rng, lo, hi)
        most = _MAX_SCORES // 3
    elif op == "kept":
        n = _length(rng, 1024, 65536)
        m = min(n, rng.choice([1, 1, 4, _log_int(rng, 16, 2048), 64 * _log_int(rng, 1, 32)]))
        out = rng.choice(["same", "fp16", "fp32"])
        b_most = 32
    else:
        use = rng.choice(["decode", "prefill", "prefill", "dropout", "total"])
        if use == "decode":
            n = _length(rng, 512, 65536)
            m = rng.choice([1, 1, 1, 2, 4, _log_int(rng, 5, 64)])
            b_most = 64
        else:
            m = n = _length(rng, lo, hi)
        if use == "prefill" and rng.random() < 0.2:
            n = _length(rng, 64, 32768)
        if use == "dropout":
            dropout, most = rng.choice([0.1, 0.2, 0.5]), 1 << 30
        if use == "total":
            total, lse, most = True, True, _MAX_SCORES // 6
        if use == "prefill":
            most = _MAX_SCORES // 3
    if m * n * h > most:  # the longest sequences with few heads
        h = hkv = 2
    while m * n * h > most:
        m = m // 2 + 1
        n = m if op != "kept" else n
    cap = min(b_most, max(1, most // (m * n * h)), max(1, (1 << 28) // (max(m, n) * h * d)))
    b = max(1, min(cap, _log_int(rng, 1, max(1.001, cap))))
    data = rng.choice(["normal", "offset", "outlier"]) if op != "flash" else "normal"
    return _case(None, op, b, h, hkv, m, n, d, dtype, layout, causal, smooth, mask, out, lse, dropout, total, data)


def _mask(c, g, dev):
    """The mask tensor of a case, or None.  Sequences are padded at the end to between half and all of the keys."""
    if c["mask"] == "none":
        return None
    kind, kind_type = c["mask"].split(":")
    b, h, m, n = c["b"], c["h"], c["m"], c["n"]
    if kind == "bias":
        return torch.randn((1, h, m, n), generator=g, device=dev).to(DTYPES[kind_type])
    lengths = n // 2 + (torch.rand((b, 1, 1, 1), generator=g, device=dev) * (n - n // 2)).long() + 1
    keep = torch.arange(n, device=dev).view(1, 1, 1, n) < lengths
    if kind == "causal_padding":
        keep = keep & (torch.arange(n, device=dev).view(1, n) <= torch.arange(m, device=dev).view(m, 1) + (n - m))
    if kind_type == "bool":
        return keep
    dt = DTYPES[kind_type]
    return torch.zeros(keep.shape, dtype=dt, device=dev).masked_fill_(~keep, torch.finfo(dt).min)


def prepare(case, seed):
    c, dev = case, torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)
    b, h, hkv, m, n, d, dt = c["b"], c["h"], c["hkv"], c["m"], c["n"], c["d"], DTYPES[c["dtype"]]
    nhd = c["layout"] == "NHD"

    def randn(heads, length):
        return torch.randn((b, length, heads, d) if nhd else (b, heads, length, d), generator=g, device=dev)

    q, k, v = randn(h, m), randn(hkv, n), randn(hkv, n)
    if c["data"] == "offset":
        k += 2.0 * torch.randn((1, 1, hkv, d) if nhd else (1, hkv, 1, d), generator=g, device=dev)
    elif c["data"] == "outlier":
        for t, heads in ((q, h), (k, hkv)):
            cols = torch.randperm(heads * d, generator=g, device=dev)[: max(1, heads * d // 100)]
            gain = torch.ones(heads * d, device=dev).index_fill_(0, cols, 20.0).view(heads, d)
            t *= gain.view(1, 1, heads, d) if nhd else gain.view(1, heads, 1, d)
        v = v.uniform_(-1.0, 1.0, generator=g)
    state = {"case": c, "q": q.to(dt), "k": k.to(dt), "v": v.to(dt), "mask": _mask(c, g, dev), "seed": seed,
             "out": dt if c["out"] == "same" else DTYPES[c["out"]]}
    if c["op"] == "kept":  # the cache holds the quantized K; the new queries come quantized from the step before
        q8, qs, k8, ks = sa.per_block_int8(state["q"], state["k"], smooth_k=True)
        state.update(q8=q8, qs=qs, k8=k8, ks=ks, q=None, k=None)
    return state


def run(state):
    c, v = state["case"], state["v"]
    if c["op"] == "step":
        q8, qs, k8, ks = sa.per_block_int8(state["q"], state["k"], tensor_layout=c["layout"], smooth_k=c["smooth"])
        o, lse = sa.sage_attention(q8, k8, v, qs, ks, tensor_layout=c["layout"], attn_mask=state["mask"],
                                   output_dtype=state["out"], return_lse=c["lse"], causal=c["causal"])
        return (o, lse) if c["lse"] else o
    if c["op"] == "sageattn":
        return sa.sageattn(state["q"], state["k"], v, is_causal=c["causal"], return_lse=c["lse"])
    if c["op"] == "kept":
        o, lse = sa.sage_attention(state["q8"], state["k8"], v, state["qs"], state["ks"], output_dtype=state["out"],
                                   return_lse=c["lse"], causal=c["causal"])
        return (o, lse) if c["lse"] else o
    if c["dropout"] > 0:
        # what recomputing activations does before it repeats a forward pass: the same state of the random stream
        torch.cuda.default_generators[v.device.index].manual_seed(state["seed"])
    res = flag_attn.flash_attention(state["q"], state["k"], v, c["causal"], dropout_p=c["dropout"],
                                    return_log_normalizer=c["lse"], return_total_attention=c["total"])
    if c["lse"] or c["total"]:
        return [t for t in res[:3] if t is not None]
    return res


def _visible_pairs(m, n, causal):
    """(query, key) pairs a head has to look at: all, or those with key <= query + (n - m)."""
    if not causal:
        return m * n
    first = n - m + 1  # keys the first query sees
    if first >= 1:
        return m * first + m * (m - 1) // 2
    return n * (n + 1) // 2


def work(case):
    """Multiply-adds of Q.K^T and P.V over the visible pairs, counted twice each; inputs read once, outputs written once."""
    c = case
    b, h, hkv, m, n, d = c["b"], c["h"], c["hkv"], c["m"], c["n"], c["d"]
    causal = c["causal"] or c["mask"].startswith("causal_padding")
    q_numel, kv_numel = b * h * m * d, b * hkv * n * d
    out_bytes = {"same": 2, "fp16": 2, "bf16": 2, "fp32": 4}[c["out"]]
    if c["op"] == "kept":
        nbytes = q_numel + 3 * kv_numel + 4 * (b * h * -(-m // 128) + b * hkv * -(-n // 64))
    else:
        nbytes = 2 * q_numel + 4 * kv_numel
    nbytes += out_bytes * q_numel + (4 * b * h * m if c["lse"] else 0) + (4 * b * h * n if c["total"] else 0)
    if c["mask"] != "none":
        kind, kind_type = c["mask"].split(":")
        entries = {"padding": b * n, "causal_padding": b * m * n, "bias": h * m * n}[kind]
        nbytes += entries * {"bool": 1, "fp32": 4}.get(kind_type, 2)
    return {"bytes": nbytes, "flops": 4 * b * h * d * _visible_pairs(m, n, causal)}


def tolerance(case):
    """Weights P and outputs are rounded to 16 bits (8 significand bits in bf16, 11 in fp16) and the sums are taken in the
    kernel's own order.  Four times what the same calls differ by from 64-bit arithmetic on the same quantized inputs,
    over the listed cases and 40 drawn ones: 2.4e-3 and 3.6e-2 with bf16, 3.0e-4 and 3.9e-3 without."""
    if "bf16" in (case["dtype"], case["out"]):
        return {"rel": 1e-2, "max": 0.15}
    return {"rel": 1.2e-3, "max": 1.6e-2}
