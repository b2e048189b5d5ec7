"""Cases that time the ring-attention path through its public entry points.

Each case is one pass of a kind of work that a program built on this package does per
layer: a causal ring prefill (contiguous, Striped / ZigZag, from a paged pool, in fp32),
a domain's ring steps with the running state, a decode step of the Q-ring, the fused
QKV projection, and the wire frames of a K/V block.  Shapes are the configurations of
bench.py and the tests (Llama-3-8B, Qwen2.5-3B and Qwen2-0.5B attention heads, uneven
domain chunks) and generic odd sizes between them.
"""
from __future__ import annotations

import importlib
import math

import numpy as np
import torch

H = importlib.import_module("hetero-cp-ringattn_amd")

DEVICE = "cuda"
TORCH_DTYPE = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
BLOCK_SIZE = 16
ROPE_BASE = 500000.0

# attention heads: query heads, KV heads, head dim (Llama-3-8B, Qwen2.5-3B, Qwen2-0.5B)
LLAMA = dict(hq=32, hkv=8, d=128)
QWEN3B = dict(hq=16, hkv=2, d=128)
QWEN05B = dict(hq=14, hkv=2, d=64)


def listed():
    return [
        # The headline workload: a 32k prompt over four uneven domains.
        dict(name="prefill_llama_32k", kind="prefill", chunks="12288,8192,8192,4096", **LLAMA, dtype="bf16",
             strategy="vanilla", paged=False),
        # An ordinary long prompt, eight query heads per KV head, three uneven domains.
        dict(name="prefill_qwen3b_8k", kind="prefill", chunks="4096,2560,1536", **QWEN3B, dtype="bf16",
             strategy="vanilla", paged=False),
        # A short chat prompt split over two domains: odd lengths, few tiles in flight.
        dict(name="prefill_llama_short", kind="prefill", chunks="517,380", **LLAMA, dtype="bf16",
             strategy="vanilla", paged=False),
        # Load-balanced (ZigZag) positions in fp16 on head dim 64, three ragged domains.
        dict(name="prefill_qwen05b_zigzag", kind="prefill", chunks="1531,1024,749", **QWEN05B, dtype="f16",
             strategy="zigzag", paged=False),
        # A prompt whose K/V live in a serving engine's paged cache: staged, then folded.
        dict(name="prefill_paged_llama_16k", kind="prefill", chunks="6144,2048,3072,5120", **LLAMA, dtype="bf16",
             strategy="vanilla", paged=True),
        # The fp32 ring of the reference's own smoke run: 1024 tokens over [640, 384].
        dict(name="prefill_f32_1k", kind="prefill", chunks="640,384", hq=8, hkv=8, d=64, dtype="f32",
             strategy="vanilla", paged=False),
        # One domain's ring steps on a continuation chunk: its own 512 tokens, then a
        # predecessor's 8192 tokens merged into the running state.
        dict(name="steps_llama_512x8k", kind="steps", lq=512, lk=8192, **LLAMA, dtype="bf16"),
        # A decode step of a full serving batch at 16k context over three growth-sharded domains.
        dict(name="decode_llama_64x16k", kind="decode", batch=64, ctx=16384, domains=3, **LLAMA, dtype="bf16",
             ragged=False),
        # A decode step of a few interactive sequences, ragged, over two domains.
        dict(name="decode_qwen3b_4x2k", kind="decode", batch=4, ctx=2085, domains=2, **QWEN3B, dtype="bf16",
             ragged=True),
        # The projection that feeds a prefill chunk's ring, rotated and appended to the paged cache.
        dict(name="qkv_llama_4096", kind="qkv", tokens=4096, hidden=4096, **LLAMA, dtype="bf16", bias=False,
             paged=True),
        # The projection of a decode step: one token of each of 64 sequences.
        dict(name="qkv_llama_64", kind="qkv", tokens=64, hidden=4096, **LLAMA, dtype="bf16", bias=False,
             paged=False),
        # A domain's K/V block to the reference's TCP payload (heads expanded to fp32) and back.
        dict(name="frame_llama_8k", kind="frame", tokens=8192, **LLAMA, dtype="bf16", expand=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _split(rng, total, n):
    """total in n uneven parts, each at least 1."""
    w = [rng.uniform(0.4, 1.6) for _ in range(n)]
    parts = [max(1, int(total * x / sum(w))) for x in w]
    parts[0] += total - sum(parts)
    return ",".join(str(p) for p in parts)


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "prefill_f32", "steps", "decode", "decode", "qkv", "qkv", "frame"])
    heads = dict(rng.choice([LLAMA, QWEN3B, QWEN05B]))
    dtype = rng.choice(["bf16", "bf16", "f16"])
    if kind == "prefill":
        s = _log_int(rng, 200, 24000)
        return dict(kind=kind, chunks=_split(rng, s, rng.randint(1, 5)), **heads, dtype=dtype,
                    strategy=rng.choice(["vanilla", "vanilla", "striped", "zigzag"]), paged=rng.random() < 0.3)
    if kind == "prefill_f32":
        s = _log_int(rng, 200, 4000)
        return dict(kind="prefill", chunks=_split(rng, s, rng.randint(1, 3)), hq=8, hkv=rng.choice([2, 8]),
                    d=rng.choice([64, 128]), dtype="f32", strategy=rng.choice(["vanilla", "zigzag"]), paged=False)
    if kind == "steps":
        return dict(kind=kind, lq=_log_int(rng, 32, 4096), lk=_log_int(rng, 256, 16384), **heads, dtype=dtype)
    if kind == "decode":
        return dict(kind=kind, batch=_log_int(rng, 1, 64), ctx=_log_int(rng, 130, 16384), domains=rng.randint(1, 4),
                    **heads, dtype=dtype, ragged=rng.random() < 0.7)
    if kind == "qkv":
        hidden = {32: 4096, 16: 2048, 14: 896}[heads["hq"]]
        return dict(kind=kind, tokens=_log_int(rng, 1, 12288), hidden=hidden, **heads, dtype=dtype,
                    bias=heads["hq"] != 32, paged=rng.random() < 0.5)
    return dict(kind="frame", tokens=_log_int(rng, 64, 12288), **heads, dtype=rng.choice(["bf16", "f16", "f32"]),
                expand=rng.random() < 0.5)


# ---------------------------------------------------------------------------------
# inputs (made from the seed alone)
# ---------------------------------------------------------------------------------
def _chunks(case):
    return [int(c) for c in case["chunks"].split(",")]


def _gen(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _normals(g, shape, dtype):
    return torch.randn(shape, generator=g, device=DEVICE, dtype=TORCH_DTYPE[dtype])


def _shard_lens(case, seed):
    """Tokens of every sequence in every domain's shard [domains][batch]: the prefill is
    split 4 : 3 : 2 : 1 and the last 5% are decode tokens owned by position mod domains."""
    n, b = case["domains"], case["batch"]
    r = np.random.default_rng(seed)
    ctx = r.integers(max(1, case["ctx"] // 2), case["ctx"] + 1, b) if case["ragged"] else np.full(b, case["ctx"])
    ctx[0] = case["ctx"]
    weights = [4, 3, 2, 1][:n]
    lens = np.zeros((n, b), np.int64)
    for i in range(b):
        pre = int(ctx[i]) - int(ctx[i]) // 20
        acc = 0
        for dom in range(n):
            part = pre - acc if dom == n - 1 else pre * weights[dom] // sum(weights)
            acc += part
            owned = sum(1 for p in range(pre, int(ctx[i])) if p % n == dom)
            lens[dom, i] = part + owned
    return lens


def _decode_inputs(case, seed):
    g = _gen(seed)
    b, d, hkv = case["batch"], case["d"], case["hkv"]
    lens = _shard_lens(case, seed)
    blocks = [int(-(-lens[dom].max() // BLOCK_SIZE)) for dom in range(case["domains"])]
    total = b * sum(blocks)
    q = _normals(g, (b, case["hq"], d), case["dtype"])
    pool = _normals(g, (2, total, BLOCK_SIZE, hkv, d), case["dtype"])
    perm = torch.randperm(total, generator=g, device=DEVICE).to(torch.int32)
    shards, cur = [], 0
    for dom in range(case["domains"]):
        table = perm[cur: cur + b * blocks[dom]].view(b, blocks[dom])
        cur += b * blocks[dom]
        shards.append((table, torch.tensor(lens[dom], dtype=torch.int32, device=DEVICE), int(lens[dom].max())))
    return q, pool, shards, lens


def _qkv_inputs(case, seed):
    g = _gen(seed)
    hidden, d, dt = case["hidden"], case["d"], case["dtype"]
    nq, nkv = case["hq"] * d, case["hkv"] * d
    x = _normals(g, (case["tokens"], hidden), dt)
    w = [_normals(g, (n, hidden), dt).mul_(1.0 / math.sqrt(hidden)) for n in (nq, nkv, nkv)]
    bias = [_normals(g, (n,), dt).mul_(0.5) for n in (nq, nkv, nkv)] if case["bias"] else [None] * 3
    if case["paged"]:
        pos = torch.arange(case["tokens"], dtype=torch.int64, device=DEVICE)
    else:
        pos = torch.randint(0, 16384, (case["tokens"],), generator=g, device=DEVICE, dtype=torch.int64)
    blocks = -(-case["tokens"] // BLOCK_SIZE)
    table = torch.randperm(blocks, generator=g, device=DEVICE).to(torch.int32)
    return x, w, bias, pos, table


def _prefill_inputs(case, seed):
    """q, then K / V as views or as a paged pool with its block table."""
    g = _gen(seed)
    s, d, hkv = sum(_chunks(case)), case["d"], case["hkv"]
    q = _normals(g, (s, case["hq"], d), case["dtype"]).permute(1, 0, 2)
    if case["paged"]:
        blocks = -(-s // BLOCK_SIZE)
        pool = _normals(g, (2, blocks, BLOCK_SIZE, hkv, d), case["dtype"])
        return q, pool, torch.randperm(blocks, generator=g, device=DEVICE).to(torch.int32)
    k = _normals(g, (s, hkv, d), case["dtype"]).permute(1, 0, 2)
    v = _normals(g, (s, hkv, d), case["dtype"]).permute(1, 0, 2)
    return q, k, v


def _steps_inputs(case, seed):
    g = _gen(seed)
    q = _normals(g, (case["lq"], case["hq"], case["d"]), case["dtype"]).permute(1, 0, 2)
    kv = [_normals(g, (n, case["hkv"], case["d"]), case["dtype"]).permute(1, 0, 2)
          for n in (case["lq"], case["lq"], case["lk"], case["lk"])]
    return q, kv


def _frame_inputs(case, seed):
    g = _gen(seed)
    shape = (case["hkv"], case["tokens"], case["d"])
    k, v = (_normals(g, shape, case["dtype"]) for _ in range(2))
    return k, v, torch.arange(4096, 4096 + case["tokens"], dtype=torch.int64, device=DEVICE)


def prepare(case, seed):
    st = {"case": case}
    if case["kind"] == "prefill":
        chunks = _chunks(case)
        q, k, v = _prefill_inputs(case, seed)
        ws = H.replay_workspace_size(q.dtype, case["hq"], case["hkv"], case["d"], chunks, paged=case["paged"],
                                     strategy=case["strategy"])
        st.update(q=q, k=k, v=v, chunks=chunks, out=torch.empty(q.shape, dtype=q.dtype, device=DEVICE),
                  lse=torch.empty(q.shape[:2], dtype=torch.float32, device=DEVICE),
                  ws=torch.empty(max(ws, 1), dtype=torch.uint8, device=DEVICE))
    elif case["kind"] == "steps":
        q, kv = _steps_inputs(case, seed)
        st.update(q=q, kv=kv, o=torch.empty(q.shape, dtype=torch.float32, device=DEVICE),
                  lse=torch.empty(q.shape[:2], dtype=torch.float32, device=DEVICE))
    elif case["kind"] == "decode":
        q, pool, shards, _ = _decode_inputs(case, seed)
        st.update(q=q, pool=pool, shards=shards, out=torch.empty_like(q),
                  lse=torch.empty(q.shape[:2], dtype=torch.float32, device=DEVICE),
                  ws=torch.empty(max(H.decode_ring_workspace_size(q, pool, shards), 1), dtype=torch.uint8,
                                 device=DEVICE))
    elif case["kind"] == "qkv":
        x, w, bias, pos, table = _qkv_inputs(case, seed)
        st.update(x=x, w=w, bias=bias, pos=pos, table=table, rope=H.rope_table(case["d"], 16384, ROPE_BASE),
                  q=torch.empty(case["hq"], x.shape[0], case["d"], dtype=x.dtype, device=DEVICE))
        if case["paged"]:
            st["pool"] = torch.zeros(2, table.numel(), BLOCK_SIZE, case["hkv"], case["d"], dtype=x.dtype,
                                     device=DEVICE)
        else:
            st["k"], st["v"] = (torch.empty(case["hkv"], x.shape[0], case["d"], dtype=x.dtype, device=DEVICE)
                                for _ in range(2))
    else:
        k, v, pos = _frame_inputs(case, seed)
        st.update(k=k, v=v, pos=pos, k2=torch.empty_like(k), v2=torch.empty_like(v), pos2=torch.empty_like(pos))
    return st


# ---------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------
def run(st):
    case = st["case"]
    if case["kind"] == "prefill":
        fn = H.ring_attention_replay_paged if case["paged"] else H.ring_attention_replay
        return fn(st["q"], st["k"], st["v"], st["chunks"], out=st["out"], lse_out=st["lse"], workspace=st["ws"],
                  strategy=case["strategy"])
    if case["kind"] == "steps":
        k0, v0, k1, v1 = st["kv"]
        H.block_partial(st["q"], k0, v0, case["lk"], case["lk"], o=st["o"], lse=st["lse"])
        return H.block_partial(st["q"], k1, v1, case["lk"], 0, o=st["o"], lse=st["lse"], accumulate=True)
    if case["kind"] == "decode":
        return H.decode_ring_replay(st["q"], st["pool"], st["shards"], 0, out=st["out"], lse_out=st["lse"],
                                    workspace=st["ws"])
    if case["kind"] == "qkv":
        (wq, wk, wv), (bq, bk, bv) = st["w"], st["bias"]
        if case["paged"]:
            q = H.qkv_rope_project_paged(st["x"], wq, wk, wv, case["hq"], case["hkv"], case["d"], st["pool"],
                                         st["table"], 0, 0, positions=st["pos"], table=st["rope"], bq=bq, bk=bk,
                                         bv=bv, q_out=st["q"])
            return q, st["pool"]
        return H.qkv_rope_project(st["x"], wq, wk, wv, case["hq"], case["hkv"], case["d"], positions=st["pos"],
                                  table=st["rope"], bq=bq, bk=bk, bv=bv, q_out=st["q"], k_out=st["k"], v_out=st["v"])
    header, payload = H.kv_frame_pack(st["k"], st["v"], 3, 4096, 4096 + case["tokens"], positions=st["pos"],
                                      num_heads=case["hq"] if case["expand"] else None)
    desc, _ = H.kv_frame_parse(header)
    desc.num_kv_heads = case["hkv"]
    H.kv_frame_unpack(desc, payload, st["k2"], st["v2"], st["pos2"])
    return np.frombuffer(header, dtype=np.uint8), payload, st["k2"], st["v2"], st["pos2"]


# ---------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------
def work(case):
    es = 4 if case["dtype"] == "f32" else 2
    d, hq, hkv = case["d"], case["hq"], case["hkv"]
    if case["kind"] == "prefill":
        s = sum(_chunks(case))
        return {"bytes": s * d * es * (2 * hq + 2 * hkv) + s * hq * 4, "flops": 2 * d * hq * s * (s + 1)}
    if case["kind"] == "steps":
        lq, lk = case["lq"], case["lk"]
        return {"bytes": lq * d * es * hq + 2 * (lq + lk) * d * es * hkv + lq * hq * (d + 1) * 4,
                "flops": 2 * d * hq * lq * (lq + 1) + 4 * d * hq * lq * lk}
    if case["kind"] == "decode":
        tokens = int(_shard_lens(case, 0).sum())
        return {"bytes": 2 * tokens * hkv * d * es + case["batch"] * hq * (2 * d * es + 4),
                "flops": 4 * tokens * hq * d}
    if case["kind"] == "qkv":
        feat = (hq + 2 * hkv) * d
        return {"bytes": es * (case["tokens"] * case["hidden"] + feat * case["hidden"] + case["tokens"] * feat),
                "flops": 2 * case["tokens"] * case["hidden"] * feat}
    wire = hq if case["expand"] else hkv
    n = 2 * case["tokens"] * d
    # pack: the block read, the payload written; unpack: one head per group read, the block written
    return {"bytes": n * hkv * es + n * wire * 4 + n * hkv * 4 + n * hkv * es + 4 * 8 * case["tokens"], "flops": 0}


def tolerance(case):
    if case["kind"] == "frame":
        return "exact"
    # four times the distance from the 64-bit result at the listed sizes: attention rounds P
    # and the output row (bf16 2.2e-3, fp16 2.6e-4), the projection its result (1.7e-3);
    # fp32 sums 2.9e-7
    return {"rel": {"bf16": 8e-3, "f16": 1e-3, "f32": 1.2e-6}[case["dtype"]]}


# ---------------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------------
def _attend(q, k, v, q_pos, k_pos):
    """Causal softmax attention of one head in fp64: q [Lq, D] against k / v [Lk, D];
    key j visible to query i iff k_pos[j] <= q_pos[i]."""
    q, k, v = q.double(), k.double(), v.double()
    s = torch.mm(q, k.t().contiguous()) / math.sqrt(q.shape[1])
    s.masked_fill_(k_pos[None, :] > q_pos[:, None], -math.inf)
    lse = torch.logsumexp(s, 1)
    return torch.mm(torch.exp_(s.sub_(lse[:, None])), v), lse


def _attend_heads(q, k, v, q_pos, k_pos):
    """[Hq, Lq, D] against [Hkv, Lk, D], 2048 query rows at a time."""
    hq, lq, d = q.shape
    rep = hq // k.shape[0]
    out = torch.empty(hq, lq, d, dtype=torch.float64, device=DEVICE)
    lse = torch.empty(hq, lq, dtype=torch.float64, device=DEVICE)
    for h in range(hq):
        for r in range(0, lq, 2048):
            rows = slice(r, min(r + 2048, lq))
            out[h, rows], lse[h, rows] = _attend(q[h, rows], k[h // rep], v[h // rep], q_pos[rows], k_pos)
    return out, lse


def exact(case, seed):
    if case["kind"] == "frame":
        return None
    if case["kind"] == "prefill":
        q, k, v = _prefill_inputs(case, seed)
        chunks = _chunks(case)
        s = sum(chunks)
        if case["paged"]:
            pool, table = k, v.long()
            k, v = (pool[i][table].reshape(-1, case["hkv"], case["d"])[:s].permute(1, 0, 2) for i in range(2))
        pos = torch.tensor(_positions(chunks, case["strategy"]), device=DEVICE)
        return _attend_heads(q, k, v, pos, pos)
    if case["kind"] == "steps":
        q, (k0, v0, k1, v1) = _steps_inputs(case, seed)
        k, v = torch.cat([k1, k0], 1), torch.cat([v1, v0], 1)
        k_pos = torch.arange(k.shape[1], device=DEVICE)
        return _attend_heads(q, k, v, k_pos[case["lk"]:], k_pos)
    if case["kind"] == "decode":
        q, pool, shards, lens = _decode_inputs(case, seed)
        rep = case["hq"] // case["hkv"]
        out = torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
        lse = torch.empty(q.shape[:2], dtype=torch.float64, device=DEVICE)
        for b in range(case["batch"]):
            kv = [torch.cat([pool[i][t[b].long()].reshape(-1, case["hkv"], case["d"])[:lens[dom, b]]
                             for dom, (t, _, _) in enumerate(shards)]) for i in range(2)]
            n = torch.arange(kv[0].shape[0], device=DEVICE)
            for h in range(case["hkv"]):
                rows = slice(h * rep, (h + 1) * rep)
                out[b, rows], lse[b, rows] = _attend(q[b, rows], kv[0][:, h], kv[1][:, h],
                                                     n[-1].expand(rep), n)
        return out, lse
    x, w, bias, pos, table = _qkv_inputs(case, seed)
    d = case["d"]
    x64 = x.double()
    # the rotation's angles are formed in fp32 (position times inverse frequency)
    inv = torch.tensor([1.0 / ROPE_BASE ** (2.0 * j / d) for j in range(d // 2)], dtype=torch.float64).float()
    ang = (pos.float()[:, None] * inv.to(DEVICE)[None, :]).double()
    cos, sin = torch.cos(ang), torch.sin(ang)
    outs = []
    for i, (wi, bi) in enumerate(zip(w, bias)):
        y = torch.mm(x64, wi.double().t().contiguous())
        if bi is not None:
            y = y + bi.double()
        y = y.view(x.shape[0], -1, d).permute(1, 0, 2)
        if i < 2:
            a, b = y[..., : d // 2], y[..., d // 2:]
            y = torch.cat([a * cos - b * sin, a * sin + b * cos], -1)
        outs.append(y)
    if not case["paged"]:
        return tuple(outs)
    pool = torch.zeros(2, table.numel() * BLOCK_SIZE, case["hkv"], d, dtype=torch.float64, device=DEVICE)
    t = torch.arange(x.shape[0], device=DEVICE)
    rows = table.long()[t // BLOCK_SIZE] * BLOCK_SIZE + t % BLOCK_SIZE
    for i in range(2):
        pool[i, rows] = outs[1 + i].permute(1, 0, 2)
    return outs[0], pool.view(2, table.numel(), BLOCK_SIZE, case["hkv"], d)


def _positions(chunks, strategy):
    """Global position of every domain-major row."""
    n, s = len(chunks), sum(chunks)
    if strategy == "vanilla":
        return list(range(s))
    owned = [[] for _ in range(n)]
    if strategy == "striped":
        # positions dealt out in turn to the domains whose chunk is not full yet
        p, left = 0, list(chunks)
        while p < s:
            for dom in range(n):
                if left[dom] > 0:
                    owned[dom].append(p)
                    left[dom] -= 1
                    p += 1
        return sum(owned, [])
    # zigzag: a prefix run of each domain in order, then the remainders in reverse order
    p = 0
    for dom in range(n):
        half = (chunks[dom] + 1) // 2
        owned[dom] += range(p, p + half)
        p += half
    for dom in reversed(range(n)):
        rest = chunks[dom] // 2
        owned[dom] += range(p, p + rest)
        p += rest
    return sum(owned, [])
