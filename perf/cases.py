"""The workloads this library is timed on, through its public entry points.

Four groups, as a decoding or prompt-processing program calls them on each
layer: the attention node on a contiguous cache, paged decode attention,
prefill attention with its cache traffic, and the k-quant projections.  A case
is a dict of plain values; "path" names the group and the rest its sizes and
options.  Inputs are drawn on the GPU from the seed alone.
"""
from __future__ import annotations

import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "nyion.rs_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "nyion.rs_amd"))

import nyion_hip as nh  # noqa: E402

KV = {"f32": nh.KV_F32, "f16": nh.KV_F16, "q4": nh.KV_Q4_20B}
FMT = {"q4k": nh.Q4K_BYTES, "q6k": nh.Q6K_BYTES}

# (heads, kv heads, head size): a 1.1B-shaped and an 8B-shaped attention, and
# the small grouped and the ungrouped head counts of the tests
GEOMETRIES = ((32, 4, 64), (32, 8, 128), (8, 2, 128), (12, 12, 64))
# rows x columns of the projections of a 1.1B- and an 8B-shaped model
LINEARS = ((2048, 2048), (256, 2048), (5632, 2048), (2048, 5632), (32000, 2048), (32003, 2048),
           (4096, 4096), (1024, 4096), (14336, 4096), (4096, 14336))
# (hidden, feed-forward, k/v width) of the two
LAYERS = ((2048, 5632, 256), (4096, 14336, 1024))

DECODE_BYTES_MAX = 2_300_000_000
PREFILL_FLOPS_MAX = 550_000_000_000
LINEAR_WORK_MAX = 509 * 5632 * 2048


def listed():
    return [
        # the attention node of a short chat turn: one call, almost no work
        dict(name="node_ctx128", path="node", kv="f32", heads=32, kv_heads=4, head_dim=64,
             ctx=128),
        # the executor's Full decode call of one sequence, with its importance
        dict(name="decode_tracked_ctx4096", path="decode", kv="f32", heads=32, kv_heads=4,
             head_dim=64, batch=1, ctx_lo=4096, ctx_hi=4096, block_tokens=16, window=0, stride=0,
             tracked=True),
        # continuous batching at its fullest, f32 cache: the headline workload
        dict(name="decode_f32_batch64", path="decode", kv="f32", heads=32, kv_heads=4,
             head_dim=64, batch=64, ctx_lo=512, ctx_hi=32768, block_tokens=16, window=0, stride=0,
             tracked=False),
        # an 8B-shaped batch on the 4-bit cache, ragged lengths
        dict(name="decode_q4_d128_batch24", path="decode", kv="q4", heads=32, kv_heads=8,
             head_dim=128, batch=24, ctx_lo=200, ctx_hi=16000, block_tokens=16, window=0,
             stride=0, tracked=False),
        # a small 8B-shaped batch of ordinary chats on the binary16 cache
        dict(name="decode_f16_d128_batch8", path="decode", kv="f16", heads=32, kv_heads=8,
             head_dim=128, batch=8, ctx_lo=300, ctx_hi=3000, block_tokens=16, window=0, stride=0,
             tracked=False),
        # long contexts under the executor's Sparse strategy (window, globals every 64)
        dict(name="decode_q4_window_ctx131072", path="decode", kv="q4", heads=32, kv_heads=4,
             head_dim=64, batch=8, ctx_lo=131072, ctx_hi=131072, block_tokens=16, window=4096,
             stride=64, tracked=False),
        # a long prompt in one call, its K/V written to f32 pages
        dict(name="prefill_8192_d128", path="prefill", kv="f32", heads=32, kv_heads=8,
             head_dim=128, rows=8192, history=0, block_tokens=16),
        # a later chunk of a chat's prompt on the 4-bit cache: history gathered,
        # attention, the chunk's K/V quantised into the cache
        dict(name="prefill_chunk_d64", path="prefill", kv="q4", heads=32, kv_heads=4, head_dim=64,
             rows=500, history=3001, block_tokens=16),
        # one token's projections of one layer, Q4_K with Q6_K v and down
        dict(name="layer_q4km_token", path="layer", mix="q4k_m", hidden=2048, ffn=5632, kv=256),
        # one token's output projection
        dict(name="linear_q6k_head_token", path="linear", fmt="q6k", rows=32000, cols=2048,
             batch=1),
        # one decode step's feed-forward projection of eight sequences, 8B-shaped
        dict(name="linear_q4k_batch8", path="linear", fmt="q4k", rows=14336, cols=4096, batch=8),
        # a prompt chunk's feed-forward projection, an odd number of tokens
        dict(name="linear_q4k_prompt", path="linear", fmt="q4k", rows=5632, cols=2048, batch=509),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("node", "decode", "decode", "decode", "prefill", "prefill", "layer",
                       "linear", "linear", "linear"))
    heads, kv_heads, head_dim = rng.choice(GEOMETRIES)
    geo = dict(heads=heads, kv_heads=kv_heads, head_dim=head_dim)
    if kind == "node":
        return dict(path="node", kv=rng.choice(("f32", "f32", "f16")), ctx=_log_int(rng, 16, 4096),
                    **geo)
    if kind == "decode":
        kv = rng.choice(("f32", "f16", "q4"))
        window = rng.choice((0, 0, 0, 256, 1024, 4096))
        tracked = window == 0 and rng.random() < 0.25
        hi = _log_int(rng, 4 * window if window else 64, 131072 if window else 32768)
        lo = max(1, int(hi * rng.choice((1.0, 0.5, 0.02))))
        c = dict(path="decode", kv=kv, batch=1, ctx_lo=lo, ctx_hi=hi,
                 block_tokens=rng.choice((16, 16, 32, 64)), window=window,
                 stride=64 if window and rng.random() < 0.7 else 0, tracked=tracked, **geo)
        held = 2 * kv_heads * hi * _row_bytes(kv, head_dim)
        c["batch"] = max(1, min(_log_int(rng, 1, 64), DECODE_BYTES_MAX // held))
        return c
    if kind == "prefill":
        rows = _log_int(rng, 32, 8192)
        history = 0 if rng.random() < 0.4 else _log_int(rng, 64, 16384)
        while 4 * heads * head_dim * rows * (history + (rows + 1) / 2) > PREFILL_FLOPS_MAX:
            history //= 2
        return dict(path="prefill", kv=rng.choice(("f32", "f16", "q4")), rows=rows,
                    history=history, block_tokens=rng.choice((16, 16, 32, 64)), **geo)
    if kind == "layer":
        hidden, ffn, kv = rng.choice(LAYERS)
        # a k/v width of its own, as grouped attention has from one kv head on
        kv = 64 * rng.randint(1, hidden // 64)
        return dict(path="layer", mix=rng.choice(("q4k", "q4k_m")), hidden=hidden, ffn=ffn, kv=kv)
    rows, cols = rng.choice(LINEARS)
    batch = max(1, min(_log_int(rng, 1, 512), LINEAR_WORK_MAX // (rows * cols)))
    return dict(path="linear", fmt=rng.choice(("q4k", "q4k", "q6k")),
                rows=max(1, rows - rng.randint(0, 40)), cols=cols, batch=batch)


# ------------------------------------------------------------------- inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def _row_bytes(kv, head_dim):
    return {"f32": 4 * head_dim, "f16": 2 * head_dim, "q4": (head_dim + 31) // 32 * 20}[kv]


def _q4_rows(x):
    """Rows of the 4-bit cache: per 32 elements a binary16 step (max|x| / 7) and
    minimum, and 16 bytes of nibbles, even elements in the low ones."""
    groups = x.reshape(-1, 32)
    d = (groups.abs().amax(1, keepdim=True) / 7).half()
    low = groups.amin(1, keepdim=True).half()
    nib = ((groups - low.float()) / d.float()).round().clamp(0, 14).to(torch.uint8)
    packed = nib[:, 0::2] | (nib[:, 1::2] << 4)
    out = torch.cat((d.view(torch.uint8), low.view(torch.uint8), packed), 1)
    return out.view(*x.shape[:-1], x.shape[-1] // 32 * 20)


def _pool(g, kv, blocks, kv_heads, block_tokens, head_dim):
    """A pool of N(0, 1) rows in the cache's format, filled in slices."""
    rows = kv_heads * block_tokens
    per = max(1, (64 << 20) // (rows * head_dim))
    parts = []
    for b in range(0, blocks, per):
        x = _normal(g, min(per, blocks - b), kv_heads, block_tokens, head_dim)
        parts.append(x if kv == "f32" else x.half() if kv == "f16" else _q4_rows(x))
    return torch.cat(parts) if len(parts) > 1 else parts[0]


def _weights(g, fmt, rows, cols):
    """A k-quant matrix as a trained one is: scales within a factor of two of
    each other, values about zero."""
    nb = cols // 256
    w = torch.randint(0, 256, (rows, nb, FMT[fmt]), dtype=torch.uint8, device="cuda", generator=g)
    d = (torch.rand((rows, nb, 1), device="cuda", generator=g) * 4.3e-4 + 7e-5).half()
    if fmt == "q4k":
        w[:, :, 0:2] = d.view(torch.uint8)
        w[:, :, 2:4] = (7.5 * d.float()).half().view(torch.uint8)
        # scales and minima 32..63: bit 5 of each six-bit field
        w[:, :, 4:12] |= 0xA0
    else:
        w[:, :, 208:210] = d.view(torch.uint8)
        sign = w[:, :, 192:208] & 0x80  # int8 scales, magnitude 64..127
        mag = (w[:, :, 192:208] & 0x3F) | 0x40
        w[:, :, 192:208] = torch.where(sign > 0, 256 - mag.short(), mag.short()).to(torch.uint8)
    return w.view(rows, nb * FMT[fmt])


def _lengths(g, c):
    lens = torch.randint(c["ctx_lo"], c["ctx_hi"] + 1, (c["batch"],), generator=g, device="cuda")
    return lens.to(torch.int32)


def _tables(g, lens, block_tokens, max_blocks):
    """Block tables of sequences that share one shuffled pool."""
    need = (lens.long() + block_tokens - 1) // block_tokens
    total = int(need.sum())
    order = torch.randperm(total, generator=g, device="cuda").to(torch.int32)
    tables = torch.zeros((len(lens), max_blocks), dtype=torch.int32, device="cuda")
    mask = torch.arange(max_blocks, device="cuda")[None, :] < need[:, None]
    tables[mask] = order
    return tables, total


def prepare(case, seed):
    nh.init(0)
    g = _generator(seed)
    c = case
    if c["path"] == "node":
        shape = (c["kv_heads"], c["ctx"], c["head_dim"])
        k, v = _normal(g, *shape), _normal(g, *shape)
        if c["kv"] == "f16":
            k, v = k.half(), v.half()
        q = _normal(g, c["heads"], c["head_dim"])
        return dict(case=c, q=q, k=k, v=v, out=torch.empty_like(q),
                    scores=torch.empty(c["heads"] * c["ctx"], device="cuda"))
    if c["path"] == "decode":
        lens = _lengths(g, c)
        max_ctx = int(lens.max())
        max_blocks = -(-max_ctx // c["block_tokens"])
        tables, blocks = _tables(g, lens, c["block_tokens"], max_blocks)
        pool = (c["kv"], blocks, c["kv_heads"], c["block_tokens"], c["head_dim"])
        k, v = _pool(g, *pool), _pool(g, *pool)
        q = _normal(g, c["batch"], c["heads"], c["head_dim"])
        s = dict(case=c, q=q, k=k, v=v, tables=tables, lens=lens, max_ctx=max_ctx,
                 out=torch.empty_like(q))
        need = nh.decode_workspace_size(c["batch"], c["heads"], c["kv_heads"], c["head_dim"],
                                        max_ctx, c["window"], c["stride"])
        s["workspace"] = nh.alloc_workspace(need)
        if c["tracked"]:
            s["scores"] = torch.empty((c["batch"], c["heads"], max_ctx + 2), device="cuda")
            s["importance"] = torch.zeros((c["batch"], max_ctx), dtype=torch.float64,
                                          device="cuda")
        else:
            s["call"] = nh.prepare_paged_decode(
                q, k, v, tables, lens, s["out"], c["heads"], c["kv_heads"], c["head_dim"],
                c["block_tokens"], max_ctx, kv_dtype=KV[c["kv"]], window=c["window"],
                global_stride=c["stride"], workspace=s["workspace"])
        return s
    if c["path"] == "prefill":
        n, hist = c["rows"], c["history"]
        lens = torch.tensor([n + hist], device="cuda", dtype=torch.int32)
        tables, blocks = _tables(g, lens, c["block_tokens"], -(-(n + hist) // c["block_tokens"]))
        q = _normal(g, n, c["heads"], c["head_dim"]).bfloat16()
        k = _normal(g, n, c["kv_heads"], c["head_dim"]).bfloat16()
        v = _normal(g, n, c["kv_heads"], c["head_dim"]).bfloat16()
        s = dict(case=c, q=q, k=k, v=v, table=tables[0], out=torch.empty(q.shape, device="cuda"))
        pool = (c["kv"], blocks, c["kv_heads"], c["block_tokens"], c["head_dim"])
        if hist:
            s["k_pool"], s["v_pool"] = _pool(g, *pool), _pool(g, *pool)
            s["k_hist"] = torch.empty((hist, c["kv_heads"], c["head_dim"]), device="cuda",
                                      dtype=torch.bfloat16)
            s["v_hist"] = torch.empty_like(s["k_hist"])
        else:
            row = _row_bytes(c["kv"], c["head_dim"])
            for name in ("k_pool", "v_pool"):
                raw = torch.zeros((blocks, c["kv_heads"], c["block_tokens"], row),
                                  dtype=torch.uint8, device="cuda")
                s[name] = (raw if c["kv"] == "q4" else
                           raw.view(torch.float32 if c["kv"] == "f32" else torch.float16))
        return s
    if c["path"] == "layer":
        hidden, ffn, kv = c["hidden"], c["ffn"], c["kv"]
        alt = "q6k" if c["mix"] == "q4k_m" else "q4k"
        h, a, m = _normal(g, hidden), _normal(g, hidden), _normal(g, ffn)
        # q, k, v | o | gate, up | down: what one layer runs between its norms
        stages = []
        for x, parts in ((h, ((hidden, "q4k"), (kv, "q4k"), (kv, alt))), (a, ((hidden, "q4k"),)),
                         (h, ((ffn, "q4k"), (ffn, "q4k"))), (m, ((hidden, alt),))):
            stages.append([(_weights(g, f, r, x.numel()), x, torch.empty(r, device="cuda"), r,
                            x.numel(), FMT[f]) for r, f in parts])
        return dict(case=c, stages=stages)
    x = _normal(g, c["batch"], c["cols"])
    return dict(case=c, x=x, w=_weights(g, c["fmt"], c["rows"], c["cols"]),
                out=torch.empty((c["batch"], c["rows"]), device="cuda"))


def run(state):
    s, c = state, state["case"]
    if c["path"] == "node":
        nh.attention_node(s["q"], s["k"], s["v"], s["out"], c["heads"], c["kv_heads"], c["ctx"],
                          c["head_dim"], c["ctx"], kv_dtype=KV[c["kv"]], scores=s["scores"])
        return s["out"]
    if c["path"] == "decode":
        if not c["tracked"]:
            s["call"]()
            return s["out"]
        nh.paged_decode_tracked(s["q"], s["k"], s["v"], s["tables"], s["lens"], s["out"],
                                s["importance"], c["heads"], c["kv_heads"], c["head_dim"],
                                c["block_tokens"], kv_dtype=KV[c["kv"]], max_ctx=s["max_ctx"],
                                workspace=s["workspace"], scores=s["scores"])
        return dict(out=s["out"], importance=s["importance"])
    if c["path"] == "prefill":
        pool = (c["block_tokens"], c["kv_heads"], c["head_dim"], KV[c["kv"]])
        into = dict(k_pool=s["k_pool"], v_pool=s["v_pool"], block_table=s["table"],
                    block_tokens=c["block_tokens"], kv_dtype=KV[c["kv"]])
        args = (s["out"], c["heads"], c["kv_heads"], c["head_dim"])
        if c["history"]:
            nh.kv_gather_bf16(s["k_pool"], s["table"], *pool, c["history"], s["k_hist"])
            nh.kv_gather_bf16(s["v_pool"], s["table"], *pool, c["history"], s["v_hist"])
            nh.prefill_bf16_ctx(s["q"], s["k"], s["v"], s["k_hist"], s["v_hist"], *args, **into)
        else:
            nh.prefill_bf16(s["q"], s["k"], s["v"], *args, **into)
        return dict(out=s["out"], k_pool=s["k_pool"], v_pool=s["v_pool"])
    if c["path"] == "layer":
        for specs in s["stages"]:
            nh.gemv_specs(specs)
        return [spec[2] for specs in s["stages"] for spec in specs]
    if c["batch"] == 1:
        gemv = nh.gemv_q4k if c["fmt"] == "q4k" else nh.gemv_q6k
        gemv(s["w"], s["x"], s["out"], c["rows"], c["cols"])
    else:
        gemv = nh.gemv_q4k_batched if c["fmt"] == "q4k" else nh.gemv_q6k_batched
        gemv(s["w"], s["x"], s["out"], c["rows"], c["cols"])
    return s["out"]


def _attended(c, ctx):
    """How many positions a sequence of ctx tokens attends to."""
    if c["window"] <= 0 or ctx - 1 <= c["window"]:
        return ctx
    start = ctx - c["window"]
    return c["window"] + (min(start // c["stride"], 128) if c["stride"] > 0 else 0)


def work(case):
    c = case
    if c["path"] == "node":
        row = _row_bytes(c["kv"], c["head_dim"])
        return {"bytes": 2 * c["kv_heads"] * c["ctx"] * row + 8 * c["heads"] * c["head_dim"],
                "flops": 4 * c["heads"] * c["head_dim"] * c["ctx"]}
    if c["path"] == "decode":
        # of the mean length: the lengths come from the seed
        tokens = c["batch"] * _attended(c, (c["ctx_lo"] + c["ctx_hi"]) // 2)
        row = _row_bytes(c["kv"], c["head_dim"])
        return {"bytes": 2 * tokens * c["kv_heads"] * row
                + 8 * c["batch"] * c["heads"] * c["head_dim"] + 4 * tokens // c["block_tokens"]
                + (16 * tokens if c["tracked"] else 0),
                "flops": 4 * c["heads"] * c["head_dim"] * tokens}
    if c["path"] == "prefill":
        n, hist, hq, hkv, d = c["rows"], c["history"], c["heads"], c["kv_heads"], c["head_dim"]
        row = _row_bytes(c["kv"], d)
        return {"bytes": n * hq * d * (2 + 4) + 2 * n * hkv * (2 * d + row) + 2 * hist * hkv * row,
                "flops": 4 * hq * d * (n * hist + n * (n + 1) // 2)}
    if c["path"] == "layer":
        per = {"q4k": 144 / 256, "q6k": 210 / 256}
        alt = per["q6k" if c["mix"] == "q4k_m" else "q4k"]
        hidden, ffn, kv = c["hidden"], c["ffn"], c["kv"]
        q4 = hidden * (2 * hidden + kv + 2 * ffn)
        rest = hidden * (kv + ffn)
        return {"bytes": int(per["q4k"] * q4 + alt * rest) + 4 * (5 * hidden + 2 * kv + 3 * ffn),
                "flops": 2 * (q4 + rest)}
    return {"bytes": c["rows"] * c["cols"] // 256 * FMT[c["fmt"]]
            + 4 * c["batch"] * (c["rows"] + c["cols"]),
            "flops": 2 * c["rows"] * c["cols"] * c["batch"]}


def tolerance(case):
    c = case
    if c["path"] == "prefill":
        return {"rel": 1e-3, "max": 2e-2}
    if c["path"] in ("node", "decode") and c["kv"] != "f32":
        return {"rel": 1e-3, "max": 2e-2}
    return {"rel": 3e-6, "max": 1e-4}


# ------------------------------------------------- the same in 64 bits

def _wide_rows(x, kv):
    """Cache rows in float64."""
    if kv != "q4":
        return x.double()
    b = x.reshape(-1, 20)
    d = b[:, 0:2].contiguous().view(torch.float16).double()
    low = b[:, 2:4].contiguous().view(torch.float16).double()
    nib = torch.stack((b[:, 4:] & 15, b[:, 4:] >> 4), 2).view(-1, 32)
    return (nib.double() * d + low).view(*x.shape[:-1], x.shape[-1] // 20 * 32)


def _wide_weights(w, fmt, rows, cols):
    """A k-quant matrix in float64."""
    b = w.view(rows * (cols // 256), FMT[fmt])
    if fmt == "q4k":
        d = b[:, 0:2].contiguous().view(torch.float16).double()
        dmin = b[:, 2:4].contiguous().view(torch.float16).double()
        s0, s1, s2 = b[:, 4:8], b[:, 8:12], b[:, 12:16]
        sc = torch.cat((s0 & 63, (s2 & 15) | ((s0 >> 6) << 4)), 1).double() * d
        mn = torch.cat((s1 & 63, (s2 >> 4) | ((s1 >> 6) << 4)), 1).double() * dmin
        qs = b[:, 16:144].reshape(-1, 4, 32)
        q = torch.stack((qs & 15, qs >> 4), 2).view(-1, 8, 32).double()
        return (q * sc[:, :, None] - mn[:, :, None]).view(rows, cols)
    d = b[:, 208:210].contiguous().view(torch.float16).double()
    sc = b[:, 192:208].contiguous().view(torch.int8).double() * d
    ql, qh = b[:, 0:128].reshape(-1, 2, 64), b[:, 128:192].reshape(-1, 2, 32)
    low = torch.cat((ql & 15, ql >> 4), 2).view(-1, 2, 4, 32)
    high = torch.stack([(qh >> (2 * k)) & 3 for k in range(4)], 2)
    q = (low | (high << 4)).double() - 32  # [block][half][k][32]
    return (q.view(-1, 16, 16) * sc[:, :, None]).view(rows, cols)


def _attend(q, k, v, causal_from=None):
    """q [H][n][D], k and v [H][t][D] in float64: the softmax average and the
    weights; row i sees keys 0 .. causal_from + i where that is given."""
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1])
    if causal_from is not None:
        n, t = s.shape[1:]
        seen = torch.arange(t, device=s.device)[None] <= torch.arange(n, device=s.device)[:, None] + causal_from
        s = s.masked_fill(~seen, -math.inf)
    p = torch.softmax(s, -1)
    return torch.matmul(p, v), p


def _sequence(pool, table, tokens, kv):
    """[kv heads][tokens][D] of one sequence in float64."""
    x = _wide_rows(pool[table[: -(-tokens // pool.shape[2])].long()], kv)
    return x.transpose(0, 1).reshape(pool.shape[1], -1, x.shape[-1])[:, :tokens].contiguous()


def exact(case, seed):
    s, c = prepare(case, seed), case
    if c["path"] in ("node", "decode"):
        group = c["heads"] // c["kv_heads"]
        shape = (c["kv_heads"], group, c["head_dim"])
        if c["path"] == "node":
            out, _ = _attend(s["q"].double().view(shape), s["k"].double(), s["v"].double())
            return out.view(s["q"].shape)
        outs = []
        weights = torch.zeros((c["batch"], s["max_ctx"]), dtype=torch.float64, device="cuda")
        for b, ctx in enumerate(s["lens"].tolist()):
            at = torch.arange(ctx, device="cuda")
            if 0 < c["window"] < ctx - 1:
                start = ctx - c["window"]
                far = min(start // c["stride"], 128) if c["stride"] > 0 else 0
                at = torch.cat((at[:far] * c["stride"], at[start:]))
            where = s["tables"][b][at // c["block_tokens"]].long(), at % c["block_tokens"]
            k, v = (_wide_rows(x[where[0], :, where[1]], c["kv"]).transpose(0, 1).contiguous()
                    for x in (s["k"], s["v"]))
            out, p = _attend(s["q"][b].double().view(shape), k, v)
            outs.append(out.view(s["q"].shape[1:]))
            weights[b, at] = p.sum((0, 1))
        out = torch.stack(outs)
        return dict(out=out, importance=weights) if c["tracked"] else out
    if c["path"] == "prefill":
        n, hist, group = c["rows"], c["history"], c["heads"] // c["kv_heads"]
        k, v = (s[x].double().transpose(0, 1) for x in ("k", "v"))
        if hist:  # attended as the caller hands it over, in bfloat16
            old = [_sequence(s[x], s["table"], hist, c["kv"]).float().bfloat16().double()
                   for x in ("k_pool", "v_pool")]
            k, v = torch.cat((old[0], k), 1), torch.cat((old[1], v), 1)
        out = torch.empty(s["out"].shape, dtype=torch.float64, device="cuda")
        for h in range(c["heads"]):
            kh = h // group
            for r in range(0, n, 2048):
                part = s["q"][r:r + 2048, h].double()
                seen = hist + min(n, r + 2048)
                out[r:r + 2048, h] = _attend(part[None], k[kh:kh + 1, :seen].contiguous(),
                                             v[kh:kh + 1, :seen].contiguous(), hist + r)[0][0]
        pools = dict(k_pool=None, v_pool=None)
        if c["kv"] != "q4":
            at = hist + torch.arange(n, device="cuda")
            blocks = s["table"][at // c["block_tokens"]].long()
            for name, x in (("k_pool", s["k"]), ("v_pool", s["v"])):
                pools[name] = s[name].double()
                pools[name][blocks, :, at % c["block_tokens"]] = x.double()
        return dict(out=out, **pools)
    if c["path"] == "layer":
        by_bytes = {n: f for f, n in FMT.items()}
        return [_wide_weights(w, by_bytes[b], r, n) @ x.double()
                for specs in s["stages"] for w, x, _, r, n, b in specs]
    wide = _wide_weights(s["w"], c["fmt"], c["rows"], c["cols"])
    return s["x"].double() @ wide.t().contiguous()
