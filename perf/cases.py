"""Performance cases of the fused attention family: what its users run, over the
sizes, types and options they run it with.

A case is a dict of plain values:
  op       the public entry point (`train`: attention forward and backward)
  B, Hq, Hk, M, N, D   batch, query heads, key/value heads, queries, keys, head dim
  dtype    "fp16" or "bf16"
  layout   "bhsd": q, k, v stored (B, H, S, D); "bshd": stored (B, S, H, D), as a
           fused QKV projection leaves them, and passed as (B, H, S, D) views
  causal, split (cross-token entry points), dropout, scale (standard deviation
  of q, k and v)
"""
from __future__ import annotations

import math

import torch

import flash_attn_with_score_amd as fas
from flash_attn_with_score_amd.attention_scores import compute_attention_scores

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}

CROSS = ("attention_cross_token_qk_sum", "attention_cross_token_softmax_sum",
         "attention_cross_token_softmax_sum_buffered")


def _case(op, B, Hq, Hk, M, N, D, dtype, causal, layout="bhsd", split=0, dropout=0.0, scale=1.0):
    return {"op": op, "B": B, "Hq": Hq, "Hk": Hk, "M": M, "N": N, "D": D, "dtype": dtype,
            "causal": causal, "layout": layout, "split": split, "dropout": dropout,
            "scale": scale}


def listed():
    named = {
        # The smallest model the family is run on: a few heads over a short
        # prompt, where the call itself is most of the time.
        "scores_tiny": _case("attention_with_scores", 1, 4, 4, 256, 256, 64, "fp16", True),
        # Attention maps of a short and a long causal prompt (analysis,
        # distillation, score-based pruning).
        "scores_1k": _case("attention_with_scores", 1, 32, 32, 1024, 1024, 128, "fp16", True),
        "scores_4k": _case("attention_with_scores", 1, 32, 32, 4096, 4096, 128, "fp16", True),
        # Attention maps of an encoder over a batch padded to its longest
        # member, whatever length that is.
        "scores_ragged": _case("attention_with_scores", 2, 16, 16, 1531, 1531, 64, "bf16", False,
                               layout="bshd"),
        # One decoding step that also updates the importance of every cached
        # key (KV-cache eviction), with a batch of grouped-query sequences.
        "decode_col_softmax": _case("attention_with_softmax_col_sum", 8, 32, 8, 1, 8191, 128,
                                    "bf16", True),
        # A short window of queries that rates a long cache (prompt
        # compression): row sums of the raw scores.
        "window_row_sum": _case("attention_with_row_sum", 1, 32, 8, 200, 8000, 128, "bf16", True),
        # Prefill of a grouped-query model with softmax column sums.
        "prefill_col_softmax": _case("attention_with_softmax_col_sum", 1, 28, 4, 4096, 4096, 128,
                                     "bf16", True),
        # Raw column sums of long sequences without a mask.
        "full_col_sum": _case("attention_with_col_sum", 2, 32, 32, 8192, 8192, 128, "fp16", False,
                              scale=0.5),
        # Cross-token sums of a long prompt against its prefix, and the two
        # others at the length a prompt more often has.
        "cross_softmax_16k": _case("attention_cross_token_softmax_sum", 1, 32, 8, 16384, 16384,
                                   128, "bf16", True, split=12288),
        "cross_qk_2k": _case("attention_cross_token_qk_sum", 1, 32, 32, 2048, 2048, 128, "fp16",
                             True, split=768),
        # Training: a causal grouped-query layer, and an encoder layer with
        # dropout over a ragged batch.
        "train_gqa": _case("train", 1, 32, 8, 4096, 4096, 128, "bf16", True, layout="bshd"),
        "train_encoder_dropout": _case("train", 4, 16, 16, 1000, 1000, 64, "fp16", False,
                                       layout="bshd", dropout=0.1),
    }
    return [dict(c, name=n) for n, c in named.items()]


OPS = ("attention_with_scores", "attention_with_row_sum", "attention_with_col_sum",
       "attention_with_col_sum_sequential", "attention_with_softmax_col_sum", *CROSS,
       "compute_attention_scores")


def _size(rng, lo, hi):
    """A size spread over [lo, hi] by its logarithm; two in five are whole
    multiples of 64, as padded batches are."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if n >= 128 and rng.random() < 0.4:
        n -= n % 64
    return n


def _cost(case):
    w = work(case)
    return w["bytes"] / 5e12 + w["flops"] / 1e15


def draw(rng):
    most = max(_cost(c) for c in listed())
    kind = rng.choice(["prefill", "prefill", "prefill", "decode", "window", "train", "train"])
    D = rng.choice([32, 64, 64, 128, 128, 128])
    dtype = rng.choice(["fp16", "bf16"])
    layout = rng.choice(["bhsd", "bshd"])
    G, Hk = rng.choice([(1, 4), (1, 12), (1, 16), (1, 32), (2, 8), (4, 8), (7, 4), (8, 4)])
    while True:
        if kind == "decode":
            op = rng.choice(["attention_with_scores", "attention_with_row_sum",
                             "attention_with_softmax_col_sum"])
            case = _case(op, rng.choice([1, 2, 4, 8, 16]), Hk * G, Hk, rng.randint(1, 8),
                         _size(rng, 256, 32768), D, dtype, True, layout)
        elif kind == "window":
            op = rng.choice(OPS[:5] + OPS[-1:])
            N = _size(rng, 512, 32768)
            case = _case(op, rng.choice([1, 1, 2]), Hk * G, Hk, _size(rng, 16, N // 4), N, D,
                         dtype, op != OPS[-1], layout)
        elif kind == "train":
            S = _size(rng, 128, 8192)
            case = _case("train", rng.choice([1, 2, 4]), Hk * G, Hk, S, S, D, dtype,
                         rng.random() < 0.7, layout, dropout=rng.choice([0.0, 0.0, 0.0, 0.1]))
        else:
            op = rng.choice(OPS)
            S = _size(rng, 128, 16384)
            causal = op != OPS[-1] and rng.random() < 0.7
            split = rng.randint(S // 8, S - S // 8) if op in CROSS else 0
            case = _case(op, rng.choice([1, 1, 2, 4]), Hk * G, Hk, S, S, D, dtype, causal, layout,
                         split=split)
        if _cost(case) <= 0.8 * most:
            return case


def _randn(gen, shape, std, dtype, layout):
    B, H, S, D = shape
    stored = (B, S, H, D) if layout == "bshd" else shape
    t = torch.randn(stored, generator=gen, device="cuda", dtype=torch.float32).mul_(std).to(dtype)
    return t.transpose(1, 2) if layout == "bshd" else t


def _inputs(case, seed):
    gen = torch.Generator("cuda").manual_seed(seed)
    c, dt = case, DTYPES[case["dtype"]]
    qs, ks = (c["B"], c["Hq"], c["M"], c["D"]), (c["B"], c["Hk"], c["N"], c["D"])
    q = _randn(gen, qs, c["scale"], dt, c["layout"])
    k = _randn(gen, ks, c["scale"], dt, c["layout"])
    v = _randn(gen, ks, c["scale"], dt, c["layout"])
    do = _randn(gen, qs, 1.0, dt, c["layout"]) if c["op"] == "train" else None
    return q, k, v, do


def prepare(case, seed):
    q, k, v, do = _inputs(case, seed)
    if do is not None:
        q, k, v = (t.requires_grad_(True) for t in (q, k, v))
    return {"case": case, "q": q, "k": k, "v": v, "do": do, "seed": seed}


def run(state):
    c, q, k, v = state["case"], state["q"], state["k"], state["v"]
    op = c["op"]
    if op == "train":
        if c["dropout"] > 0:
            # A step that can be repeated starts its random stream itself.
            torch.cuda.manual_seed(state["seed"])
        o = fas.attention(q, k, v, causal=c["causal"], dropout_p=c["dropout"])
        dq, dk, dv = torch.autograd.grad(o, (q, k, v), state["do"])
        return {"o": o, "dq": dq, "dk": dk, "dv": dv}
    if op == "compute_attention_scores":
        return {"scores": compute_attention_scores(q, k)}
    fn = getattr(fas, op)
    if op in CROSS:
        o, side = fn(q, k, v, c["split"], causal=c["causal"])
    else:
        o, side = fn(q, k, v, causal=c["causal"])
    return {"o": o, "side": side}


def _pairs(case, row_lo=0, key_hi=None):
    """Admissible (query, key) pairs of one head with query >= row_lo, key < key_hi."""
    M, N = case["M"], case["N"]
    hi = N if key_hi is None else key_hi
    if not case["causal"]:
        return (M - row_lo) * hi
    # Query i sees keys j <= i + N - M (M <= N in every case).
    first, last = row_lo + N - M + 1, N  # keys that the first and last query see
    ramp = max(0, min(last, hi) - first + 1)  # queries that see first .. min(last, hi) keys
    count = M - row_lo
    return (first + min(last, hi)) * ramp // 2 + (count - ramp) * hi


def work(case):
    B, Hq, Hk, M, N, D = (case[x] for x in ("B", "Hq", "Hk", "M", "N", "D"))
    op, e = case["op"], 2
    heads, q, kv = B * Hq, e * B * Hq * M * D, e * B * Hk * N * D
    if op == "compute_attention_scores":
        return {"bytes": q + kv + e * heads * M * N, "flops": 2 * heads * D * M * N}
    pairs = _pairs(case)
    if op == "train":
        # q, k, v, dO in; O, dQ, dK, dV out (O stays for the backward).
        return {"bytes": 4 * q + 4 * kv, "flops": 14 * heads * D * pairs}
    moved, flops = 2 * q + 2 * kv, 4 * heads * D * pairs
    if op == "attention_with_scores":
        moved += e * heads * M * N
    elif op == "attention_with_row_sum":
        moved += 4 * heads * M
    else:
        moved += 4 * B * Hk * (case["split"] or N)
    if op == "attention_with_softmax_col_sum":
        flops += 2 * heads * D * pairs
    elif op in CROSS[1:]:
        flops += 2 * heads * D * _pairs(case, case["split"], case["split"])
    return {"bytes": moved, "flops": flops}


# Results are rounded to 16 bits, and so are the softmax weights on their way
# into the second product (and dS in the backward pass), as the entry points
# promise.  2-norm errors against 64 bits, measured: fp16 2.1e-4 to 3.0e-4,
# bf16 1.7e-3 to 2.5e-3; four times the largest.
REL = {"fp16": 1.2e-3, "bf16": 1e-2}


def tolerance(case):
    return {"rel": REL[case["dtype"]]}


def _keep(case, seed, b, h):
    """The dropout mask of one head: weight (b, h, i, j) is kept where Philox
    4x32 of 6 rounds (Salmon, Moraes, Dror, Shaw, SC'11) under the generator's
    seed, at the weight's linear index, gives a uniform above p."""
    M, N = case["M"], case["N"]
    low = 0xFFFFFFFF
    start = (b * case["Hq"] + h) * M * N
    c0 = torch.arange(start, start + M * N, device="cuda", dtype=torch.int64) & low
    c1, c2, c3 = (torch.zeros_like(c0) for _ in range(3))
    k0, k1 = seed & low, (seed >> 32) & low

    def product(m, x):  # the two 32-bit halves of m * x
        a, b0 = m * (x >> 16), m * (x & 0xFFFF)
        mid = (a & 0xFFFF) * 65536 + b0
        return ((a >> 16) + (mid >> 32)) & low, mid & low

    for _ in range(6):
        h0, l0 = product(0xD2511F53, c0)
        h2, l2 = product(0xCD9E8D57, c2)
        c0, c1, c2, c3 = h2 ^ c1 ^ k0, l2, h0 ^ c3 ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & low, (k1 + 0xBB67AE85) & low
    x = torch.where(c0 >= 2**31, 2**32 - 1 - c0, c0)
    return (x.to(torch.float32) * 4.6566127342e-10 > case["dropout"]).view(M, N)


def exact(case, seed):
    q, k, v, do = _inputs(case, seed)
    B, Hq, Hk, M, N, D = (case[x] for x in ("B", "Hq", "Hk", "M", "N", "D"))
    op, split, G, sm = case["op"], case["split"], Hq // Hk, 1.0 / math.sqrt(D)
    f8 = {"device": "cuda", "dtype": torch.float64}
    if op == "train":
        out = {"o": torch.empty(B, Hq, M, D, **f8), "dq": torch.empty(B, Hq, M, D, **f8),
               "dk": torch.zeros(B, Hk, N, D, **f8), "dv": torch.zeros(B, Hk, N, D, **f8)}
    elif op == "compute_attention_scores":
        out = {"scores": torch.empty(B, Hq, M, N, **f8)}
    elif op == "attention_with_scores":
        out = {"o": torch.empty(B, Hq, M, D, **f8), "side": torch.empty(B, Hq, M, N, **f8)}
    elif op == "attention_with_row_sum":
        out = {"o": torch.empty(B, Hq, M, D, **f8), "side": torch.empty(B, Hq, M, **f8)}
    else:
        out = {"o": torch.empty(B, Hq, M, D, **f8),
               "side": torch.zeros(B, Hk, split or N, **f8)}
    # Blocks of query rows bound the memory of the longest sequences.
    step = M if op == "train" else min(M, 4096)
    for b in range(B):
        for h in range(Hq):
            kd, vd = k[b, h // G].double(), v[b, h // G].double()
            for r in range(0, M, step):
                rows = slice(r, min(M, r + step))
                qd = q[b, h, rows].double()
                s = (qd @ kd.t()) * sm
                if op == "compute_attention_scores":
                    out["scores"][b, h, rows] = s
                    continue
                hidden = None
                if case["causal"]:
                    i = torch.arange(rows.start, rows.stop, device="cuda")[:, None] + N - M
                    hidden = torch.arange(N, device="cuda")[None, :] > i
                p = s if hidden is None else s.masked_fill(hidden, float("-inf"))
                p = torch.softmax(p, dim=-1)
                raw = s if hidden is None else s.masked_fill_(hidden, 0.0)
                if op == "train":
                    z = 1.0
                    if case["dropout"] > 0:
                        z = _keep(case, seed, b, h).double() / (1.0 - case["dropout"])
                    dod = do[b, h].double()
                    pz = p * z
                    o = pz @ vd
                    out["o"][b, h] = o
                    out["dv"][b, h // G] += pz.t() @ dod
                    ds = p * ((dod @ vd.t()) * z - (dod * o).sum(-1, keepdim=True)) * sm
                    out["dq"][b, h] = ds @ kd
                    out["dk"][b, h // G] += ds.t() @ qd
                    continue
                out["o"][b, h, rows] = p @ vd
                lo = min(max(split - rows.start, 0), raw.shape[0])  # rows before the split
                if op == "attention_with_scores":
                    out["side"][b, h, rows] = raw
                elif op == "attention_with_row_sum":
                    out["side"][b, h, rows] = raw.sum(-1)
                elif op == CROSS[0]:
                    out["side"][b, h // G] += raw[lo:, :split].sum(0)
                elif op in CROSS[1:]:
                    out["side"][b, h // G] += p[lo:, :split].sum(0)
                elif op == "attention_with_softmax_col_sum":
                    out["side"][b, h // G] += p.sum(0)
                else:
                    out["side"][b, h // G] += raw.sum(0)
    return out
