"""The calls that the speed of this library is measured on.

Twelve listed cases, each a call that programs built on the library make, and
`draw`, which makes further cases of the same twelve kinds over the sizes,
ragged ones among them, that each kind is used at. Every case goes through the
Python entry points `attention_fwd` and `qk_score_tile` on device tensors.

The library is a forward-only attention library: its directions are prefill
(many query rows), decode (one or a few query rows against a long cache) and
the score tile without the softmax. Its data types are fp32 (the type of the
C++ interface it is a drop-in for), bf16 and fp16.
"""

from __future__ import annotations

import math
import os
import sys

import torch

# The package directory is not a Python identifier; the working folder is the
# repository's root.
_PKG = os.path.join(os.getcwd(), "dnn-flash_amd", "python")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import onednn_flash_hip as F  # noqa: E402

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def _attention(name, dtype, batch, heads, queries, keys, dim, value_dim=0, causal=False, layout="bhtd",
               bias="none", softcap=0.0, mask="none", algorithm="auto", std=1.0):
    case = {"name": name, "op": "attention", "dtype": dtype, "batch": batch, "heads": heads,
            "queries": queries, "keys": keys, "dim": dim, "value_dim": value_dim or dim, "causal": causal,
            "layout": layout, "bias": bias, "softcap": softcap, "mask": mask, "algorithm": algorithm,
            "std": std}
    if not name:
        del case["name"]
    return case


def _score(name, dtype, tiles, queries, keys, dim, bias="none", softcap=0.0):
    case = {"name": name, "op": "score", "dtype": dtype, "tiles": tiles, "queries": queries, "keys": keys,
            "dim": dim, "bias": bias, "softcap": softcap}
    if not name:
        del case["name"]
    return case


def listed():
    return [
        # The smallest call: one short fp32 sequence, non-causal, as an encoder
        # layer of a small model makes it. Latency and launches count.
        _attention("fp32_small", "f32", 1, 4, 512, 512, 64),
        # An fp32 decoder layer's prefill at an ordinary size, causal.
        _attention("fp32_causal", "f32", 2, 8, 2048, 2048, 64, causal=True),
        # fp32 decoding of a batch of sequences: one new row per sequence
        # against its cache of keys and values.
        _attention("fp32_decode", "f32", 16, 16, 1, 4096, 64),
        # standard_attention, the exact two-pass entry that programs compare
        # against, causal; also where head widths end that the matrix-core
        # kernels do not take (drawn below).
        _attention("fp32_standard", "f32", 2, 8, 1024, 1024, 64, causal=True, algorithm="rowwise"),
        # The headline: a large bf16 batch in causal prefill.
        _attention("bf16_prefill", "bf16", 4, 32, 4096, 4096, 128, causal=True),
        # One prompt of ordinary, ragged length through a 32-head layer, in the
        # [B, T, H, D] storage that a fused QKV projection leaves.
        _attention("bf16_prompt", "bf16", 1, 32, 1000, 1000, 128, causal=True, layout="bthd"),
        # bf16 decoding of one sequence with eight heads against a long cache.
        _attention("bf16_decode", "bf16", 1, 8, 1, 32768, 128),
        # A long bidirectional layer with ALiBi and a soft-cap: every score
        # modification at once, and the largest work of the list.
        _attention("bf16_alibi_softcap", "bf16", 2, 16, 8192, 8192, 128, bias="alibi", softcap=50.0),
        # A long document with a causal sliding window of 16 blocks of 64 keys
        # and four blocks that every row sees.
        _attention("fp16_blocksparse", "f16", 1, 16, 16384, 16384, 64, causal=True, mask="window", std=0.5),
        # A layer with a learned position bias [M, N] that all heads share.
        _attention("fp16_bias", "f16", 2, 16, 2048, 2048, 64, bias="shared"),
        # Score tiles in the exact fp32 order (bit-identical with the
        # sequential sum), for programs that run a softmax of their own.
        _score("score_fp32", "f32", 32, 1024, 1024, 128),
        # The same in bf16 with a bias that all tiles share.
        _score("score_bf16_bias", "bf16", 32, 2048, 2048, 128, bias="shared"),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw(rng):
    kind = rng.choice(["fp32_small", "fp32_causal", "fp32_decode", "fp32_standard", "bf16_prefill",
                       "bf16_prompt", "bf16_decode", "bf16_alibi_softcap", "fp16_blocksparse",
                       "fp16_bias", "score_fp32", "score_bf16_bias"])
    layout = rng.choice(["bhtd", "bthd"])
    if kind == "fp32_small":  # short sequences, few heads, every width up to 128
        m = _log(rng, 16, 1024)
        n = m if rng.random() < 0.6 else _log(rng, 16, 1024)
        return _attention("", "f32", rng.choice([1, 1, 2]), rng.choice([1, 2, 4, 8]), m, n,
                          rng.choice([32, 48, 64, 64, 80, 128]), causal=rng.random() < 0.3, layout=layout)
    if kind == "fp32_causal":  # ordinary fp32 prefill, causal or not
        n = _log(rng, 700, 4096)
        return _attention("", "f32", rng.choice([1, 2, 4]), rng.choice([4, 8, 12, 16]), n, n,
                          rng.choice([32, 64, 64, 96, 128]), causal=rng.random() < 0.7, layout=layout)
    if kind == "fp32_decode":
        return _attention("", "f32", _log(rng, 1, 32), rng.choice([4, 8, 12, 16]), rng.choice([1, 1, 1, 2, 5]),
                          _log(rng, 200, 16384), rng.choice([64, 64, 80, 128]), layout=layout)
    if kind == "fp32_standard":
        # standard_attention at any width, or a width that is no multiple of
        # the 16-byte chunk (50, 75, 100 ...), which takes the same kernel
        n = _log(rng, 64, 1100)
        odd = rng.random() < 0.5
        dtype = rng.choice(["f32", "f32", "bf16", "f16"]) if odd else "f32"
        dim = rng.choice([20, 36, 50, 75, 100] if dtype != "f32" else [25, 50, 75, 97]) if odd else \
            rng.choice([32, 64, 64, 80, 128])
        return _attention("", dtype, rng.choice([1, 2]), rng.choice([2, 4, 8]), n,
                          n if rng.random() < 0.7 else _log(rng, 64, 1100), dim, causal=rng.random() < 0.5,
                          layout=layout, algorithm="auto" if odd else "rowwise")
    if kind == "bf16_prefill":  # large prefill
        n = _log(rng, 2048, 8192)
        return _attention("", rng.choice(["bf16", "bf16", "f16"]), rng.choice([1, 2, 4, 8]),
                          rng.choice([16, 24, 32]), n, n, rng.choice([64, 128, 128, 128]),
                          causal=rng.random() < 0.75, layout=layout)
    if kind == "bf16_prompt":  # one prompt or a small batch; encoders and cross-attention
        n = _log(rng, 40, 3000)
        causal = rng.random() < 0.6
        m = n if causal or rng.random() < 0.6 else _log(rng, 40, 3000)
        dim, dv = rng.choice([(64, 64), (64, 64), (80, 80), (128, 128), (128, 128), (128, 128), (256, 256),
                              (192, 128)])
        return _attention("", rng.choice(["bf16", "bf16", "f16"]), _log(rng, 1, 8), rng.choice([8, 12, 16, 32]),
                          m, n, dim, dv, causal=causal, layout=layout)
    if kind == "bf16_decode":
        return _attention("", rng.choice(["bf16", "bf16", "f16"]), _log(rng, 1, 64), rng.choice([8, 16, 32]),
                          rng.choice([1, 1, 1, 2, 4, 16]), _log(rng, 300, 65536), rng.choice([64, 128, 128, 128]),
                          layout=layout)
    if kind == "bf16_alibi_softcap":
        n = _log(rng, 512, 8192)
        bias, softcap = rng.choice([("alibi", 50.0), ("alibi", 0.0), ("none", 30.0)])
        return _attention("", rng.choice(["bf16", "bf16", "f16"]), rng.choice([1, 2]), rng.choice([8, 16, 32]),
                          n, n, rng.choice([64, 128, 128]), causal=rng.random() < 0.5, layout=layout, bias=bias,
                          softcap=softcap)
    if kind == "fp16_blocksparse":
        n = _log(rng, 1500, 16384)
        return _attention("", rng.choice(["f16", "bf16"]), rng.choice([1, 1, 2]), rng.choice([8, 16]), n, n,
                          rng.choice([64, 64, 128]), causal=True, layout=layout, mask="window", std=0.5)
    if kind == "fp16_bias":
        m = _log(rng, 128, 4096)
        n = m if rng.random() < 0.6 else _log(rng, 128, 4096)
        return _attention("", rng.choice(["f16", "bf16"]), rng.choice([1, 2, 4]), rng.choice([8, 12, 16]), m, n,
                          rng.choice([64, 64, 128]), causal=m == n and rng.random() < 0.3, layout=layout,
                          bias=rng.choice(["shared", "shared", "per_head"]))
    if kind == "score_fp32":
        m = _log(rng, 64, 1200)
        n = m if rng.random() < 0.5 else _log(rng, 64, 1200)
        return _score("", "f32", _log(rng, 4, 32), m, n, rng.choice([32, 64, 64, 96, 100, 128]),
                      bias=rng.choice(["none", "shared", "per_tile"]))
    m = _log(rng, 128, 2500)
    n = m if rng.random() < 0.5 else _log(rng, 128, 2500)
    return _score("", rng.choice(["bf16", "f16"]), _log(rng, 4, 48), m, n, rng.choice([64, 80, 128, 128]),
                  bias=rng.choice(["none", "shared", "shared", "per_tile"]),
                  softcap=rng.choice([0.0, 0.0, 0.0, 30.0]))


def draw(rng):
    # no drawn case does more than the largest listed one of its speed
    while True:
        case = _draw(rng)
        w = work(case)
        exact_order = case["op"] == "score" and case["dtype"] == "f32"
        two_pass = case["op"] == "attention" and (case["algorithm"] == "rowwise" or _odd_width(case))
        limit = 8.6e9 if exact_order else 2.2e9 if two_pass else 1.1e11 if case["dtype"] == "f32" else 9e11
        if w["flops"] <= limit and w["bytes"] <= 5.4e8:
            return case


def _odd_width(case):
    chunk = 4 if case["dtype"] == "f32" else 8
    return case["dim"] % chunk != 0 or case["value_dim"] % chunk != 0


def _window_mask(tokens):
    """64x64 blocks: a causal window of 16 blocks plus the first four."""
    nb = (tokens + 63) // 64
    qb, kb = torch.arange(nb)[:, None], torch.arange(nb)[None, :]
    return ((kb <= qb) & ((qb - kb < 16) | (kb < 4))).to(torch.uint8)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, std=1.0, dtype=torch.float32):
        return (torch.randn(shape, device="cuda", generator=gen) * std).to(dtype)

    dtype = DTYPES[case["dtype"]]
    m, n, d = case["queries"], case["keys"], case["dim"]
    if case["op"] == "score":
        t = case["tiles"]
        bias = {"none": None, "shared": (m, n), "per_tile": (t, m, n)}[case["bias"]]
        return {"op": "score", "q": normal(t, m, d, dtype=dtype), "k": normal(t, n, d, dtype=dtype),
                "options": {"scale": 1.0 / math.sqrt(d), "bias": None if bias is None else normal(*bias),
                            "softcap": case["softcap"]}}
    b, h, dv = case["batch"], case["heads"], case["value_dim"]

    def tokens(count, width):
        if case["layout"] == "bthd":
            return normal(b, count, h, width, std=case["std"], dtype=dtype).transpose(1, 2)
        return normal(b, h, count, width, std=case["std"], dtype=dtype)

    options = {"scale": 1.0 / math.sqrt(d), "causal": case["causal"], "softcap": case["softcap"]}
    state = {"op": "attention", "q": tokens(m, d), "k": tokens(n, d), "v": tokens(n, dv), "options": options}
    if case["bias"] == "alibi":
        slopes = [2.0 ** (-8.0 * (i + 1) / h) for i in range(h)]
        options["alibi_slopes"] = torch.tensor(slopes, device="cuda", dtype=torch.float32)
    elif case["bias"] == "shared":
        options["bias"] = normal(m, n)
    elif case["bias"] == "per_head":
        options["bias"] = normal(b, h, m, n)
    if case["mask"] == "window":
        options["mask"] = _window_mask(n).cuda()
        options["mask_block_size"] = (64, 64)
    if case["algorithm"] == "rowwise":
        options["algorithm"] = F.ALGO_ROWWISE
    return state


def run(state):
    if state["op"] == "score":
        return F.qk_score_tile(state["q"], state["k"], **state["options"])
    return F.attention_fwd(state["q"], state["k"], state["v"], **state["options"])


def _pairs(case):
    """Query-key pairs of one head that no rule masks."""
    m, n = case["queries"], case["keys"]
    if case["op"] == "score" or not case["causal"]:
        return m * n
    if case["mask"] == "none":
        return sum(min(n, i + 1) for i in range(m))
    total = 0
    for i in range(m):  # rows of block qb see the first four blocks and 16 up to their own
        qb = i // 64
        last = i + 1
        first = max(0, (qb - 15) * 64)
        total += last - first + min(first, 256)
    return total


def work(case):
    es = 4 if case["dtype"] == "f32" else 2
    m, n, d = case["queries"], case["keys"], case["dim"]
    if case["op"] == "score":
        t = case["tiles"]
        bias = {"none": 0, "shared": m * n, "per_tile": t * m * n}[case["bias"]]
        return {"bytes": t * (m + n) * d * es + 4 * t * m * n + 4 * bias, "flops": 2 * t * m * n * d}
    bh, dv = case["batch"] * case["heads"], case["value_dim"]
    bias = {"none": 0, "alibi": case["heads"], "shared": m * n, "per_head": bh * m * n}[case["bias"]]
    if case["causal"] and case["bias"] in ("shared", "per_head"):
        bias = bias // (m * n) * _pairs(case)
    mask = ((n + 63) // 64) ** 2 if case["mask"] == "window" else 0
    # with a causal rule, keys past the last query row are never needed
    seen = min(m, n) if case["causal"] else n
    return {"bytes": bh * (m * d + seen * d + seen * dv + m * dv) * es + 4 * bias + mask,
            "flops": 2 * (d + dv) * _pairs(case) * bh}


def tolerance(case):
    """The relative errors against 64 bits that the measurements showed, times about four."""
    if case["op"] == "score":
        if case["dtype"] == "f32":
            return "exact"  # the sequential fp32 sum, one rounding per product and per add
        return {"rel": 5e-7}  # exact products, fp32 sums in any order
    return {"rel": {"f32": 4e-6, "f16": 1.2e-3, "bf16": 1e-2}[case["dtype"]]}


def exact(case, seed):
    state = prepare(case, seed)
    opt = state["options"]
    if state["op"] == "score":
        s = torch.empty(state["q"].shape[0], case["queries"], case["keys"], dtype=torch.float64, device="cuda")
        for t in range(s.shape[0]):
            s[t] = state["q"][t].double() @ state["k"][t].double().t().contiguous() * opt["scale"]
            if opt["bias"] is not None:
                s[t] += opt["bias"].double() if opt["bias"].dim() == 2 else opt["bias"][t].double()
            if opt["softcap"] > 0.0:
                s[t] = opt["softcap"] * torch.tanh(s[t] / opt["softcap"])
        return s
    m, n = case["queries"], case["keys"]
    out = torch.empty(case["batch"], case["heads"], m, case["value_dim"], dtype=torch.float64, device="cuda")
    rows = max(1, min(m, (1 << 26) // n))  # rows of scores formed at once
    i_all, j = torch.arange(m, device="cuda"), torch.arange(n, device="cuda")
    blocks = opt["mask"].bool() if "mask" in opt else None
    for b in range(case["batch"]):
        for h in range(case["heads"]):
            kt = state["k"][b, h].double().t().contiguous()
            v = state["v"][b, h].double()
            for r0 in range(0, m, rows):
                i = i_all[r0:r0 + rows]
                s = state["q"][b, h, r0:r0 + rows].double() @ kt * opt["scale"]
                if "alibi_slopes" in opt:
                    s += opt["alibi_slopes"][h].double() * (j[None, :] - i[:, None])
                if "bias" in opt:
                    s += (opt["bias"] if opt["bias"].dim() == 2 else opt["bias"][b, h])[r0:r0 + rows].double()
                if opt["softcap"] > 0.0:
                    s = opt["softcap"] * torch.tanh(s / opt["softcap"])
                if opt["causal"]:
                    s.masked_fill_(j[None, :] > i[:, None], -math.inf)
                if blocks is not None:
                    s.masked_fill_(~blocks[i // 64][:, j // 64], -math.inf)
                out[b, h, r0:r0 + rows] = torch.softmax(s, dim=-1) @ v
    return out
