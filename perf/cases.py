"""The work that a user of the paged KV cache has it do, as cases that can be timed and
compared: decode steps and prompt chunks of one layer (and a batched step of several), the
block-table gather and the attention prelude, over the range of sizes, batch shapes, storage
types and query groups that a serving program meets.

A case is a dict of plain values:
  op        "decode", "prefill", "gather" or "prelude"
  dtype     the pool's storage, "f16" or "q8_0"
  kv_heads, group (query heads per KV head), head_dim, block
  seqs, layers           the batch: one item per (sequence, layer)
  ctx_min, ctx_max       positions that each sequence holds before the chunk or after the step
  tok_min, tok_max       prefill: new tokens of each sequence
  norm                   prelude: the QK norm
"""
import math
import random

import torch

from qubivex_amd import HipDevice, KvLayout

_device = None


def device():
    """The program's one device handle."""
    global _device
    if _device is None:
        _device = HipDevice(0)
    return _device


def _case(op, name=None, dtype="f16", kv_heads=8, group=4, head_dim=128, block=16, seqs=1, layers=1,
          ctx=(0, 0), tok=(0, 0), norm="none"):
    c = {"op": op, "dtype": dtype, "kv_heads": kv_heads, "group": group, "head_dim": head_dim,
         "block": block, "seqs": seqs, "layers": layers, "ctx_min": ctx[0], "ctx_max": ctx[1],
         "tok_min": tok[0], "tok_max": tok[1], "norm": norm}
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # A chat turn of a small model (16 layers, 8 KV heads of 64): one sequence's decode
        # step on one layer, the smallest call, where launches and latency count.
        _case("decode", "decode_one_short", head_dim=64, ctx=(640, 640)),
        # One long document in an otherwise idle server: a decode step on one layer with a
        # single sequence, where the context has to be spread over the chip.
        _case("decode", "decode_one_long", kv_heads=4, group=8, ctx=(32768, 32768)),
        # Batched decode in model order: one layer of 32 ragged sequences.
        _case("decode", "decode_ragged", seqs=32, ctx=(256, 4096)),
        # The same with a quantised pool: one layer of 64 sequences of 2048 positions.
        _case("decode", "decode_q8", dtype="q8_0", seqs=64, ctx=(2048, 2048)),
        # Serving scale (4 KV heads, 8 query heads each): 128 sequences of 8192 positions, two
        # layers' items in one call.
        _case("decode", "decode_batch", kv_heads=4, group=8, seqs=128, layers=2, ctx=(8192, 8192)),
        # A new prompt of a small model: 512 tokens from position 0, one layer.
        _case("prefill", "prompt_short", head_dim=64, tok=(512, 512)),
        # Prompts whose prefix the prefix cache holds: a few new tokens each over a shared
        # 2047-token prefix, ragged.
        _case("prefill", "prefix_hits", seqs=8, ctx=(2047, 2047), tok=(8, 64)),
        # One request's prompt in chunks: 512 tokens at 8 k positions, one layer.
        _case("prefill", "chunk_one", kv_heads=4, group=8, ctx=(8192, 8192), tok=(512, 512)),
        # Chunks of many requests at serving scale: the largest call.
        _case("prefill", "chunk_batch", kv_heads=4, group=8, seqs=24, ctx=(7679, 7679), tok=(512, 512)),
        # The same with a quantised pool at 2 k positions.
        _case("prefill", "chunk_q8", dtype="q8_0", seqs=16, ctx=(1535, 1535), tok=(512, 512)),
        # A layer's cache read back as f32 from a quantised pool (a host model's own attention).
        _case("gather", "gather_q8", dtype="q8_0", seqs=64, ctx=(1024, 2048)),
        # The prelude of a prompt chunk with per-head QK norms and rotary positions.
        _case("prelude", "prelude_heads", kv_heads=4, group=8, tok=(8192, 8192), norm="per_head"),
    ]


# The largest listed cases bound what a drawn case may cost.
_MOST_FLOPS, _MOST_BYTES = 1.6e12, 4.0e9


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the kinds of calls above over the sizes between them, odd ones too."""
    while True:
        kind = rng.choice(["decode"] * 5 + ["prefill"] * 5 + ["gather", "prelude"])
        c = _case(kind, dtype=rng.choice(["f16", "f16", "q8_0"]), kv_heads=rng.choice([2, 4, 8, 8]),
                  group=rng.choice([1, 2, 4, 4, 7, 8, 8, 16]), head_dim=rng.choice([64, 128, 128]),
                  block=rng.choice([16, 16, 16, 32, 256]))
        if kind == "decode" or kind == "gather":
            c["seqs"] = _log(rng, 1, 128)
            c["layers"] = rng.choice([1, 1, 1, 2])
            c["ctx_max"] = _log(rng, 64, 32768)
            c["ctx_min"] = rng.choice([c["ctx_max"], c["ctx_max"] // 2 + 1, c["ctx_max"] // 16 + 1])
        elif kind == "prefill":
            c["seqs"] = _log(rng, 1, 24)
            c["tok_max"] = _log(rng, 4, 1024)
            c["tok_min"] = rng.choice([c["tok_max"], c["tok_max"] // 2 + 1, c["tok_max"] // 8 + 1])
            c["ctx_max"] = rng.choice([0, _log(rng, 32, 16384), _log(rng, 32, 16384)])
            c["ctx_min"] = rng.choice([c["ctx_max"], c["ctx_max"] // 2])
        else:
            c["dtype"], c["block"] = "f16", 16
            c["tok_max"] = c["tok_min"] = _log(rng, 16, 16384)
            c["norm"] = rng.choice(["none", "per_head", "per_head", "full"])
        w = work(c)
        if w["flops"] <= _MOST_FLOPS and w["bytes"] <= _MOST_BYTES:
            return c


# ---- what a case's sizes come to ----

def _lens(c):
    """(context, new tokens) of each sequence, the same for every seed: for a decode step or a
    gather the positions held, for a chunk the positions before it and its tokens."""
    r = random.Random(c["ctx_min"] * 7919 + c["ctx_max"] * 31 + c["tok_max"])
    ctx = [r.randint(c["ctx_min"], c["ctx_max"]) for _ in range(c["seqs"])]
    tok = [r.randint(c["tok_min"], c["tok_max"]) for _ in range(c["seqs"])]
    return ctx, tok


def work(c):
    """Each input read once, each output written once; the matrix work of Q.K and P.V."""
    G, D, H = c["kv_heads"], c["head_dim"], c["kv_heads"] * c["group"]
    row = 2 * G * D * (2 if c["dtype"] == "f16" else 34 / 32)  # a stored key and value row
    items = c["seqs"] * c["layers"]
    ctx, tok = (c["ctx_min"] + c["ctx_max"]) / 2, (c["tok_min"] + c["tok_max"]) / 2
    if c["op"] == "decode":  # stored rows, q, out, the new rows in and into the pool
        return {"bytes": items * (ctx * row + 2 * H * D * 4 + 2 * G * D * 4),
                "flops": items * 4.0 * H * D * ctx}
    if c["op"] == "prefill":
        return {"bytes": items * ((ctx + 2 * tok) * row + tok * (2 * H * D * 4 + 2 * G * D * 4)),
                "flops": items * 4.0 * H * D * tok * (ctx + (tok + 1) / 2)}
    if c["op"] == "gather":
        return {"bytes": items * ctx * (row + 2 * G * D * 4), "flops": 0.0}
    # prelude: q and k in place, the rotary rows (v passes through unchanged)
    return {"bytes": tok * (2 * (H + G) * D * 4 + D * 4), "flops": 10.0 * tok * (H + G) * D}


def tolerance(c):
    if c["op"] in ("gather", "prelude"):
        return "exact"  # the path's own rule: bytes and bits, whatever the kernel
    # about four times what the path's own alternatives (other splits of the context, the
    # probabilities carried exactly) differ by
    if c["op"] == "prefill" and c["dtype"] == "f16":
        # probabilities enter P.V as one f16 each (relative 2^-11), so two correct kernels
        # whose running maxima differ round them differently
        return {"rel": 8e-4, "max": 1e-2}
    if c["dtype"] == "q8_0":
        # a probability times its value scale is an f16 and an f16 residual, which loses
        # bits where the product is small against the running maximum's
        return {"rel": 8e-5, "max": 2.5e-3} if c["op"] == "prefill" else {"rel": 4e-5, "max": 1.2e-3}
    return {"rel": 1e-5, "max": 4e-4}  # f32 sums in another order


# ---- the pool's contents, from the seed alone ----

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _rows(c, lens, seed):
    """The stored rows, item after item, in pieces: (first row, k, v), each [n, G * D]."""
    n, kv = sum(lens), c["kv_heads"] * c["head_dim"]
    gen, step = _gen(seed * 3 + 1), max(1, (64 << 20) // kv)
    for r0 in range(0, n, step):
        shape = (min(step, n - r0), kv)
        pair = []
        for _ in range(2):
            x = torch.randn(shape, generator=gen, device="cuda")
            if c["dtype"] == "q8_0":  # 1 % outliers, which widen a group's scale
                x = torch.where(torch.rand(shape, generator=gen, device="cuda") < 0.01, 8 * x, x)
            pair.append(x)
        yield r0, pair[0], pair[1]


def _stored(c, x):
    """Rows as the pool holds them, in 64 bits."""
    if c["dtype"] == "f16":
        return x.half().double()
    g = x.reshape(-1, 32)
    d = g.abs().amax(1, keepdim=True)
    d = d / torch.full_like(d, 127.0)  # (by a scalar it would be a multiplication)
    inv = torch.where(d > 0, torch.ones_like(d) / d, torch.zeros_like(d))
    y = (g * inv).double()
    q = (torch.sign(y) * torch.floor(y.abs() + 0.5)).clamp(-127, 127)
    return (q * d.half().double()).reshape(x.shape)


def _i32(x):
    return x.to(torch.int32)


class _Batch:
    """A pool filled with the items' rows through shuffled block tables, and the tables.  The
    last `new[i]` rows of item i are the pass's own: kept in k, v (with their slots), not stored."""

    def __init__(self, c, lens, new, seed):
        self.case, self.dev, self.lens = c, device(), lens
        self.layout = KvLayout(c["dtype"], c["kv_heads"], c["head_dim"], c["block"])
        self.heads = c["kv_heads"] * c["group"]
        B = c["block"]
        n = torch.tensor(lens, dtype=torch.int64, device="cuda")
        need = (n + B - 1) // B
        at = torch.cumsum(need, 0) - need
        self.n_blocks = int(need.sum()) * 5 // 4 + 16
        perm = torch.randperm(self.n_blocks, generator=_gen(seed * 3 + 2), device="cuda")
        self.tables = perm[: int(need.sum())]
        self.blocks, self.table_at = _i32(self.tables), _i32(at)
        self.pool = torch.zeros(self.n_blocks * self.layout.block_bytes // 4, dtype=torch.int32,
                                device="cuda")
        item = torch.repeat_interleave(torch.arange(len(lens), device="cuda"), n)
        p = torch.arange(int(n.sum()), device="cuda") - (torch.cumsum(n, 0) - n)[item]
        self.slots = _i32(self.tables[at[item] + p // B] * B + p % B)
        fresh = p >= (n - torch.tensor(new, dtype=torch.int64, device="cuda"))[item]
        kept = ([], [])
        for r0, k, v in _rows(c, lens, seed):
            f, s = fresh[r0:r0 + k.shape[0]], self.slots[r0:r0 + k.shape[0]]
            for x, y in zip(kept, (k, v)):
                x.append(y[f])
            k, v, s = k[~f], v[~f], s[~f]
            if s.numel():
                self.dev.append(self.layout, self.pool, self.n_blocks, k, v, s)
        self.k, self.v = (torch.cat(x) for x in kept)
        self.new_slots = self.slots[fresh]

    def randn(self, seed, *shape):
        return torch.randn(shape, generator=_gen(seed), device="cuda")


def prepare(c, seed):
    ctx, tok = _lens(c)
    G, D = c["kv_heads"], c["head_dim"]
    H = G * c["group"]
    if c["op"] == "prelude":
        gen = _gen(seed * 3)
        s = tok[0]
        q, k, v = (torch.randn((s, n * D), generator=gen, device="cuda") for n in (H, G, G))
        ang = torch.rand((s, D // 2), generator=gen, device="cuda") * 6.2831853
        st = {"case": c, "q": q, "k": k, "v": v, "rope": torch.cat([ang.cos(), ang.sin()], 1).contiguous()}
        n = {"none": (0, 0), "per_head": (D, D), "full": (H * D, G * D)}[c["norm"]]
        st["q_norm"], st["k_norm"] = ((1 + 0.1 * torch.randn(x, generator=gen, device="cuda")) if x else None
                                      for x in n)
        st["layout"] = KvLayout(c["dtype"], G, D, c["block"])
        return st
    lens = [a + b for a, b in zip(ctx, tok)] * c["layers"]
    st = {"case": c}
    new = {"decode": [1] * len(lens), "prefill": tok * c["layers"], "gather": [0] * len(lens)}[c["op"]]
    b = st["batch"] = _Batch(c, lens, new, seed)
    n, t = (torch.tensor(x, dtype=torch.int64, device="cuda") for x in (lens, new))
    if c["op"] != "gather":
        st["q"] = b.randn(seed * 3, sum(new), H, D)
        st["out"] = torch.empty_like(st["q"])
        st["max_pos"] = max(lens) - 1
    if c["op"] == "decode":
        st["pos"] = _i32(n - 1)
    elif c["op"] == "prefill":
        st["pos0"], st["n_tok"], st["q_at"] = _i32(n - t), _i32(t), _i32(torch.cumsum(t, 0) - t)
        st["max_tok"] = max(tok)
    else:
        st["item_lens"], st["out_at"] = _i32(n), torch.cumsum(n, 0) - n
        st["max_len"] = max(lens)
        st["out_k"], st["out_v"] = (torch.empty(sum(lens) * G * D, device="cuda") for _ in range(2))
    return st


def run(st):
    c = st["case"]
    dev = device()
    if c["op"] == "prelude":
        dev.prelude(st["layout"], c["kv_heads"] * c["group"], st["q"], st["k"], st["v"], st["rope"],
                    norm=c["norm"], q_norm=st["q_norm"], k_norm=st["k_norm"])
        return {"q": st["q"], "k": st["k"], "v": st["v"]}
    b = st["batch"]
    if c["op"] == "decode":
        dev.append_attention(b.layout, b.pool, b.n_blocks, st["q"], b.k, b.v, b.blocks,
                             b.table_at, st["pos"], b.heads, st["max_pos"], st["out"])
        return {"out": st["out"], "pool": b.pool}
    if c["op"] == "prefill":
        dev.append(b.layout, b.pool, b.n_blocks, b.k, b.v, b.new_slots)
        dev.prefill_attention(b.layout, b.pool, b.n_blocks, st["q"], b.blocks, b.table_at, st["pos0"],
                              st["q_at"], st["n_tok"], b.heads, st["max_pos"], st["max_tok"], st["out"])
        return {"out": st["out"], "pool": b.pool}
    dev.gather(b.layout, b.pool, b.n_blocks, b.blocks, b.table_at, st["item_lens"], st["out_at"],
               st["max_len"], st["out_k"], st["out_v"])
    return {"k": st["out_k"], "v": st["out_v"]}


# ---- the same in 64 bits, in plain torch ----

def _attend(q, k, v, first):
    """q [t, group, D], token j at position first + j; k, v [n, D]: softmax attention of the
    tokens over the positions up to their own."""
    t, group, D = q.shape
    s = torch.matmul(q.reshape(t * group, D), k.t().contiguous()).reshape(t, group, -1) / math.sqrt(D)
    if t > 1:
        n = torch.arange(k.shape[0], device="cuda")
        s.masked_fill_((n[None, :] > first + torch.arange(t, device="cuda")[:, None])[:, None, :], -math.inf)
    p = torch.softmax(s, 2)
    return torch.matmul(p.reshape(t * group, -1), v).reshape(t, group, D)


def exact(c, seed):
    ctx, tok = _lens(c)
    G, D, gs = c["kv_heads"], c["head_dim"], c["group"]
    if c["op"] == "prelude":
        st = prepare(c, seed)
        cos, sin = st["rope"].double()[:, None, :D // 2], st["rope"].double()[:, None, D // 2:]
        out = {"v": st["v"].double()}
        for name, heads in (("q", G * gs), ("k", G)):
            x = st[name].double().reshape(-1, heads, D)
            if c["norm"] != "none":
                w = st[name + "_norm"].double()
                over = (2,) if c["norm"] == "per_head" else (1, 2)
                x = x / torch.sqrt(x.square().mean(over, keepdim=True) + 1e-6)
                x = x * (w if c["norm"] == "per_head" else w.reshape(heads, D))
            a, b = x[..., :D // 2], x[..., D // 2:]
            out[name] = torch.cat([a * cos - b * sin, a * sin + b * cos], 2).reshape(-1, heads * D)
        return out
    lens = [a + b for a, b in zip(ctx, tok)] * c["layers"]
    if c["op"] == "gather":
        outs = {"k": [], "v": []}
        rows = {"k": [], "v": []}
        for _, k, v in _rows(c, lens, seed):
            rows["k"].append(_stored(c, k).float())  # an f32 holds these values exactly
            rows["v"].append(_stored(c, v).float())
        for name in outs:
            x, at = torch.cat(rows[name]).reshape(-1, G, D), 0
            for n in lens:
                outs[name].append(x[at:at + n].transpose(0, 1).reshape(-1).double())
                at += n
        return {name: torch.cat(x) for name, x in outs.items()}
    toks = (tok if c["op"] == "prefill" else [1] * c["seqs"]) * c["layers"]
    q = torch.randn((sum(toks), G * gs, D), generator=_gen(seed * 3), device="cuda").double()
    out = torch.empty_like(q)
    pieces = _rows(c, lens, seed)
    held, at, r = None, 0, 0
    for n, t in zip(lens, toks):
        while held is None or held[0].shape[0] < n:  # the rows of the next item
            _, k, v = next(pieces)
            more = (_stored(c, k), _stored(c, v))
            held = more if held is None else tuple(torch.cat(x) for x in zip(held, more))
        k, v = (x[:n].reshape(n, G, D).transpose(0, 1).contiguous() for x in held)
        held = tuple(x[n:] for x in held)
        for g in range(G):
            step = max(1, (1 << 28) // (n * gs))
            for j in range(0, t, step):
                qq = q[r + j:r + min(t, j + step), g * gs:(g + 1) * gs]
                out[r + j:r + min(t, j + step), g * gs:(g + 1) * gs] = _attend(qq, k[g], v[g], n - t + j)
        r += t
    return {"out": out, "pool": None}
