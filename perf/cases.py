"""Measured cases of the Gated DeltaNet path: one linear-attention layer's call
in each phase a serving engine runs it in, through the backends' ``forward``
(and the layer, and the LogState reconstruction), with the metadata a program
prepares once per batch and reuses for every layer already in hand.

Sizes are those of the benchmark (``bench.py``: 16 key / 32 value heads of
128 channels, conv width 4, 1024-token checkpoint pages, 256-token LogState
pages of granularity 32) and of the tests (odd lengths, smaller head groups,
f16 io, io-typed pools).

``exact`` restates each call in float64 torch; the io-dtype roundings that
are part of the operators' definition (conv pre-activation and output, the
normalised q and k of the prefill) are kept, everything else is unrounded.
"""

import math
from types import SimpleNamespace

import numpy as np
import torch

from logssms_amd.cache import LinearStatePool
from logssms_amd.core import Batch, Context, LogStateCacheMetadata, Request, set_global_ctx
from logssms_amd.kernel.linear_attention import restore_log_state_chains
from logssms_amd.layers import GatedDeltaConfig, GatedDeltaLogStateBackend, GatedDeltaNet

DEV = "cuda"
W = 4  # conv width
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
LS_PAGE, LS_GRAN, LS_FRAME = 256, 32, 65536
HIDDEN = 2048


def _heads(hk=16, hv=32, dim=128):
    return {"heads_k": hk, "heads_v": hv, "dim": dim}


def listed():
    full = _heads()
    return [
        # one user's next token: latency and launch cost, 4 MiB of traffic
        {"name": "decode_1", "op": "decode", "batch": 1, "slots": 64, "io": "bf16", "state": "f32", **full},
        # an ordinary, odd decode batch in f16 with an f16 pool (the reference's single-dtype pool)
        {"name": "decode_37_f16", "op": "decode", "batch": 37, "slots": 256, "io": "f16", "state": "f16", **full},
        # the decode benchmark: 256 sequences in a pool of 1024 slots
        {"name": "decode_256", "op": "decode", "batch": 256, "slots": 1024, "io": "bf16", "state": "f32", **full},
        # the speculative-verify benchmark: 64 sequences of 8 drafts, every step's state kept
        {"name": "verify_64x8", "op": "verify", "batch": 64, "drafts": 8, "io": "bf16", "state": "f32", **full},
        # a short prompt on its own
        {"name": "prefill_1x300", "op": "prefill", "seqs": 1, "tokens": 300, "skew": 0.0, "hits": 0.0, "page": 1024,
         "io": "bf16", "state": "f32", **full},
        # one long prompt resuming from a cached prefix, a checkpoint per page
        {"name": "prefill_1x8192_hit", "op": "prefill", "seqs": 1, "tokens": 8192, "skew": 0.0, "hits": 1.0,
         "page": 1024, "io": "bf16", "state": "f32", **full},
        # the prefill benchmark: 4 x 4096 tokens
        {"name": "prefill_4x4096", "op": "prefill", "seqs": 4, "tokens": 16384, "skew": 0.0, "hits": 0.0,
         "page": 4096, "io": "bf16", "state": "f32", **full},
        # the packed varlen benchmark: lognormal lengths, half of the sequences from cached prefixes
        {"name": "prefill_64_varlen", "op": "prefill", "seqs": 64, "tokens": 147612, "skew": 1.0, "hits": 0.5,
         "page": 1024, "io": "bf16", "state": "f32", **full},
        # LogState decode: 256 sequences at random page positions (0..15 replayed tokens)
        {"name": "ls_decode_256", "op": "ls_decode", "batch": 256, **full},
        # LogState prefill of a few ragged prompts, every token logged
        {"name": "ls_prefill_3_ragged", "op": "ls_prefill", "seqs": 3, "tokens": 6001, "skew": 0.7, **full},
        # LogState reconstruction: 128 chains of a base state and one logged page
        {"name": "ls_restore_128", "op": "ls_restore", "chains": 128, "logged": 256, **full},
        # the whole layer (projections, GDN, gated norm, output projection) on two prompts
        {"name": "layer_2x1500", "op": "layer", "seqs": 2, "tokens": 3000, "skew": 0.0, "hits": 0.0, "page": 1024,
         "io": "bf16", "state": "f32", **full},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    heads = rng.choice([_heads(), _heads(), _heads(8, 16, 128), _heads(4, 4, 64)])
    io = rng.choice(["bf16", "bf16", "f16"])
    state = rng.choice(["f32", "f32", io])
    op = rng.choice(["decode", "verify", "prefill", "prefill", "prefill", "ls_decode", "ls_prefill", "ls_restore",
                     "layer"])
    if op == "decode":
        batch = _log_int(rng, 1, 256)
        return {"op": op, "batch": batch, "slots": batch + rng.randrange(32, 768), "io": io, "state": state, **heads}
    if op == "verify":
        return {"op": op, "batch": _log_int(rng, 1, 64), "drafts": rng.randint(2, 8), "io": io, "state": state,
                **heads}
    if op == "prefill":
        seqs = _log_int(rng, 1, 64)
        tokens = _log_int(rng, max(64, 16 * seqs), min(8192 * seqs, 140000))
        return {"op": op, "seqs": seqs, "tokens": tokens, "skew": rng.choice([0.0, 0.5, 1.0]),
                "hits": rng.choice([0.0, 0.5, 1.0]), "page": rng.choice([256, 1024]), "io": io, "state": state,
                **heads}
    if op == "ls_decode":
        return {"op": op, "batch": _log_int(rng, 1, 256), **_heads()}
    if op == "ls_prefill":
        seqs = _log_int(rng, 1, 8)
        return {"op": op, "seqs": seqs, "tokens": _log_int(rng, 40 * seqs, 4096 * seqs), "skew": 0.7, **_heads()}
    if op == "ls_restore":
        return {"op": op, "chains": _log_int(rng, 1, 128), "logged": rng.randint(16, 256), **_heads()}
    seqs = rng.randint(1, 4)
    return {"op": op, "seqs": seqs, "tokens": _log_int(rng, 64 * seqs, 2048 * seqs), "skew": 0.5, "hits": 0.0,
            "page": 1024, "io": "bf16", "state": "f32", **_heads()}


# ------------------------------------------------------------------ shared inputs

def _lengths(c):
    """Sequence lengths of a case: equal parts (skew 0) or lognormal ones,
    scaled to the case's token count, 16..16384 each."""
    n, total = c["seqs"], c["tokens"]
    if c["skew"] == 0.0 or n == 1:
        return [total // n + (i < total % n) for i in range(n)]
    rng = np.random.default_rng(1000 * n + total)
    share = rng.lognormal(0.0, c["skew"], n)
    lens = np.clip(np.rint(share * (total / share.sum())), 16, 16384).astype(int)
    i = 0
    while lens.sum() != total:  # the rounding and clipping remainder, spread over the sequences
        step = int(np.sign(total - lens.sum())) * max(1, abs(int(total - lens.sum())) // n)
        lens[i % n] = min(16384, max(16, lens[i % n] + step))
        i += 1
    return lens.tolist()


def _config(c, layer=0):
    hk, hv, d = c["heads_k"], c["heads_v"], c["dim"]
    return GatedDeltaConfig(hk, hv, d, d, 2 * hk * d + hv * d, W - 1, layer)


def _conv_dim(c):
    return (2 * c["heads_k"] + c["heads_v"]) * c["dim"]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, dtype=torch.float32, std=1.0):
    x = torch.empty(*shape, device=DEV, dtype=torch.float32).normal_(0.0, std, generator=g)
    return x.to(dtype)


def _inputs(c, rows, g, io):
    """Projections and layer weights: mixed_qkv, gate, beta, conv weight, A_log, dt_bias."""
    hv, C = c["heads_v"], _conv_dim(c)
    s = SimpleNamespace()
    s.mixed = torch.empty(rows, C, device=DEV, dtype=io)
    for a in range(0, rows, 16384):  # in pieces: the fp32 draw of the largest case would take 5 GB at once
        b = min(rows, a + 16384)
        s.mixed[a:b] = _randn(g, b - a, C)
    s.gate = _randn(g, rows, hv, dtype=io)
    s.beta = _randn(g, rows, hv, dtype=io)
    s.weight = _randn(g, C, 1, W, dtype=io, std=0.3)
    s.A_log = -torch.rand(hv, device=DEV, generator=g)
    s.dt_bias = _randn(g, hv, std=0.5)
    return s


def _pool(c, slots, g, io):
    hk, hv, d = c["heads_k"], c["heads_v"], c["dim"]
    pool = LinearStatePool(slots, 1, _conv_dim(c), W, hv, d, d, torch.device(DEV), io, DTYPES[c["state"]])
    pool.recurrent_state.normal_(0.0, 0.1, generator=g)
    pool.conv_state.normal_(0.0, 1.0, generator=g)
    return pool


# ------------------------------------------------------------------ prepare

def prepare(case, seed):
    return {"decode": _prepare_decode, "verify": _prepare_verify, "prefill": _prepare_prefill,
            "layer": _prepare_layer, "ls_decode": _prepare_ls_decode, "ls_prefill": _prepare_ls_prefill,
            "ls_restore": _prepare_ls_restore}[case["op"]](case, seed)


def _prepare_decode(c, seed):
    g, io = _gen(seed), DTYPES[c["io"]]
    b = c["batch"]
    s = _inputs(c, b, g, io)
    s.pool = _pool(c, c["slots"], g, io)
    slots = torch.randperm(c["slots"], generator=g, device=DEV)[:b].to(torch.int32)
    ctx = Context(page_size=64, linear_state=s.pool, state_table=slots[:, None].expand(b, 64).contiguous())
    s.batch = Batch(reqs=[Request(i, 30, 31) for i in range(b)], phase="decode")
    _bind(c, s, ctx)
    return s


def _prepare_verify(c, seed):
    g, io = _gen(seed), DTYPES[c["io"]]
    b, t = c["batch"], c["drafts"]
    s = _inputs(c, b * t, g, io)
    slots = 2 * b * (t + 1)
    s.pool = _pool(c, slots, g, io)
    perm = torch.randperm(slots, generator=g, device=DEV).to(torch.int32)
    ctx = Context(page_size=64, linear_state=s.pool, state_table=perm[:b, None].expand(b, 64).contiguous(),
                  work_state_table=perm[b:b + b * t].view(b, t).contiguous())
    s.batch = Batch(reqs=[Request(i, 30, 30 + t) for i in range(b)], phase="verify")
    _bind(c, s, ctx)
    return s


def _prefill_batch(c, g, io):
    """Pool, slot table and batch of a prefill: cached prefixes are one page,
    every page of a sequence has a slot of its own."""
    lens, page = _lengths(c), c["page"]
    hits = round(c["hits"] * len(lens))
    cached = [page if i < hits else 0 for i in range(len(lens))]
    counts = [-(-(n + k) // page) for n, k in zip(lens, cached)]
    slots = sum(counts)
    perm = torch.randperm(slots, generator=g, device=DEV).to(torch.int32)
    width = max(counts)
    table = torch.full((len(lens), width), -1, dtype=torch.int32, device=DEV)
    at = 0
    for r, k in enumerate(counts):
        table[r, :k] = perm[at:at + k]
        at += k
    pool = _pool(c, slots, g, io)
    ctx = Context(page_size=page, linear_state=pool, state_table=table.repeat_interleave(page, 1))
    batch = Batch(reqs=[Request(i, k, k + n) for i, (n, k) in enumerate(zip(lens, cached))], phase="prefill")
    return pool, ctx, batch


def _prepare_prefill(c, seed):
    g, io = _gen(seed), DTYPES[c["io"]]
    s = _inputs(c, c["tokens"], g, io)
    s.pool, ctx, s.batch = _prefill_batch(c, g, io)
    _bind(c, s, ctx)
    return s


def _prepare_layer(c, seed):
    g, io = _gen(seed), DTYPES[c["io"]]
    s = SimpleNamespace(op=c["op"])
    s.net = GatedDeltaNet(HIDDEN, c["heads_k"], c["heads_v"], c["dim"], c["dim"], W, 1e-6, 0, device=DEV, dtype=io)
    for t in (s.net.in_proj_qkvz_weight, s.net.in_proj_ba_weight, s.net.out_proj_weight):
        t.copy_(_randn(g, *t.shape, dtype=io, std=0.02))
    s.net.conv1d_weight.copy_(_randn(g, *s.net.conv1d_weight.shape, dtype=io, std=0.3))
    s.net.A_log.uniform_(-1.0, 0.0, generator=g)
    s.net.dt_bias.copy_(_randn(g, c["heads_v"], dtype=io, std=0.5))
    s.x = _randn(g, c["tokens"], HIDDEN, dtype=io)
    s.pool, s.ctx, s.batch = _prefill_batch(c, g, io)
    s.ctx.batch = s.batch
    s.ctx.linear_attn_backend.prepare_metadata(s.batch)
    return s


def _bind(c, s, ctx):
    s.op, s.cfg, s.ctx = c["op"], _config(c), ctx
    s.backend = ctx.linear_attn_backend
    s.backend.prepare_metadata(s.batch)


def _ls_pool(c, works, logs, g):
    """A LogState frame storage: slots 0..works-1 hold states, the next
    ``logs`` slots one page's token log each.  Each kind of frame fills one
    span of the storage, in random order: states, logs, decay records, conv
    snapshots."""
    hk, hv, d = c["heads_k"], c["heads_v"], c["dim"]
    C = _conv_dim(c)
    head = d * d * 2
    state_frames = -(-hv * head // LS_FRAME)
    log_frames = -(-2 * LS_PAGE * (hk + hv) * d // LS_FRAME)
    record = 4 * LS_PAGE * hv
    per = LS_FRAME // record
    slots, grans = works + logs, LS_PAGE // LS_GRAN
    conv_frames = -(-2 * C * (W - 1) // LS_FRAME)
    dec = -(-slots // per)
    ends = np.cumsum([works * state_frames, logs * log_frames, dec, slots * grans * conv_frames]).tolist()

    def order(a, b):
        return (torch.randperm(b - a, generator=g, device=DEV) + a).to(torch.int32)

    payload = torch.full((slots, max(state_frames, log_frames)), -1, dtype=torch.int32, device=DEV)
    payload[:works, :state_frames] = order(0, ends[0]).view(works, -1)
    payload[works:, :log_frames] = order(ends[0], ends[1]).view(logs, -1)
    dframes = order(ends[1], ends[2])
    ids = torch.arange(slots, device=DEV)
    storage = torch.empty(ends[3], LS_FRAME, dtype=torch.uint8, device=DEV)
    parts = SimpleNamespace(states=storage[:ends[0]].view(torch.bfloat16),
                            logs=storage[ends[0]:ends[1]].view(torch.bfloat16),
                            decays=storage[ends[1]:ends[2]].view(torch.float32),
                            conv=storage[ends[2]:].view(torch.bfloat16))
    parts.states.normal_(0.0, 0.1, generator=g)
    parts.logs.normal_(0.0, d ** -0.5, generator=g)  # unit keys, residuals of the same size
    parts.decays.uniform_(-0.7, 0.0, generator=g)
    parts.conv.normal_(0.0, 1.0, generator=g)
    layout = SimpleNamespace(head_k_dim=d, head_v_dim=d, num_value_heads=hv, num_key_heads=hk, num_linear_layers=1,
                             granularity=LS_GRAN, log_decay_bytes=record, num_granules=grans, conv_dim=C,
                             state_len=W - 1)
    pool = SimpleNamespace(
        storage=storage, dtype=torch.bfloat16, frame_bytes=LS_FRAME, head_payload_bytes=head, page_size=LS_PAGE,
        payload_frame_table=payload, decay_frame_table=torch.stack([dframes[ids // per], (ids % per).int()], 1),
        conv_frame_table=order(ends[2], ends[3]).view(slots, grans, conv_frames), layout=layout, parts=parts,
        allocator=SimpleNamespace(slot=lambda i: SimpleNamespace(kind="work" if i < works else "log")))
    elems = torch.arange(C * (W - 1), device=DEV)

    def read_conv(slot, granule, layer):  # windows [n, C, W - 1] of the (slot, granule) snapshots
        assert conv_frames == 1 and layer == 0
        fr = pool.conv_frame_table[slot.long().clamp_min(0), granule.long(), 0].long()
        rows = storage.view(torch.bfloat16).view(-1)[fr[:, None] * (LS_FRAME // 2) + elems].view(-1, C, W - 1)
        return torch.where((slot >= 0)[:, None, None], rows, torch.zeros((), dtype=rows.dtype, device=DEV))

    pool.read_conv = read_conv
    return pool


def _prepare_ls_decode(c, seed):
    g, b = _gen(seed), c["batch"]
    s = _inputs(c, b, g, torch.bfloat16)
    s.pool = _ls_pool(c, b, b, g)
    pos = torch.randint(0, LS_PAGE, (b,), generator=g, device=DEV, dtype=torch.int32)
    s.positions = pos
    ids = torch.arange(b, dtype=torch.int32, device=DEV)
    ctx = Context(page_size=LS_PAGE, linear_state=s.pool, work_state_table=ids[:, None],
                  state_table=(b + ids)[:, None].expand(b, LS_PAGE).contiguous(),
                  page_table=torch.arange(LS_PAGE, dtype=torch.int32, device=DEV).repeat(b, 1))
    host = pos.tolist()
    s.batch = Batch(reqs=[Request(i, p, p + 1) for i, p in enumerate(host)], phase="decode", positions=pos,
                    out_loc=pos, cache_metadata=LogStateCacheMetadata(replay_counts=[p % 16 for p in host]))
    _bind_ls(c, s, ctx)
    return s


def _prepare_ls_prefill(c, seed):
    g = _gen(seed)
    s = _inputs(c, c["tokens"], g, torch.bfloat16)
    lens = _lengths(c)
    n, width = len(lens), -(-max(lens) // LS_PAGE)
    pages = [-(-k // LS_PAGE) for k in lens]
    s.pool = _ls_pool(c, 2 * n, sum(pages), g)
    table = torch.full((n, width), -1, dtype=torch.int32, device=DEV)
    at = 2 * n
    writes, end = [], 0
    for r, (k, m) in enumerate(zip(lens, pages)):
        table[r, :m] = torch.arange(at, at + m, dtype=torch.int32, device=DEV)
        at += m
        if k >= LS_PAGE:  # a checkpoint state at the last page boundary, into a work slot of its own
            writes.append((end + k // LS_PAGE * LS_PAGE - 1, n + r))
        end += k
    pos = torch.cat([torch.arange(k, dtype=torch.int32, device=DEV) for k in lens])
    ctx = Context(page_size=LS_PAGE, linear_state=s.pool, state_table=table.repeat_interleave(LS_PAGE, 1),
                  work_state_table=torch.arange(n, dtype=torch.int32, device=DEV)[:, None],
                  page_table=torch.arange(width * LS_PAGE, dtype=torch.int32, device=DEV).repeat(n, 1))
    s.batch = Batch(reqs=[Request(i, 0, k) for i, k in enumerate(lens)], phase="prefill", positions=pos, out_loc=pos,
                    cache_metadata=LogStateCacheMetadata(first_offsets=[0] * n, checkpoint_writes=writes))
    # the prompts start from empty states and histories
    s.pool.parts.states.zero_()
    s.pool.parts.conv.zero_()
    _bind_ls(c, s, ctx)
    return s


def _bind_ls(c, s, ctx):
    s.op, s.cfg, s.ctx = c["op"], _config(c), ctx
    s.backend = GatedDeltaLogStateBackend(ctx)
    s.backend.prepare_metadata(s.batch)


def _prepare_ls_restore(c, seed):
    g, n = _gen(seed), c["chains"]
    s = SimpleNamespace(op=c["op"])
    s.pool = _ls_pool(c, 2 * n, n, g)
    s.tasks = [(i, [(2 * n + i, 0, c["logged"])], n + i) for i in range(n)]
    return s


# ------------------------------------------------------------------ run

def run(s):
    if s.op == "layer":
        set_global_ctx(s.ctx)
        out = s.net.forward(s.x)
        return {"out": out, "states": s.pool.recurrent_state, "conv": s.pool.conv_state}
    if s.op == "ls_restore":
        restore_log_state_chains(s.pool, s.tasks)
        return {"states": s.pool.parts.states}
    out = s.backend.forward(s.mixed, s.gate, s.beta, s.weight, s.A_log, s.dt_bias, s.cfg, s.batch)
    if s.op in ("ls_decode", "ls_prefill"):
        p = s.pool.parts
        return {"out": out, "states": p.states, "logs": p.logs, "decays": p.decays, "conv": p.conv}
    return {"out": out, "states": s.pool.recurrent_state, "conv": s.pool.conv_state}


# ------------------------------------------------------------------ work, tolerance

def work(c):
    hk, hv, d = c["heads_k"], c["heads_v"], c["dim"]
    C = _conv_dim(c)
    window = C * (W - 1) * 2
    token = 2 * C + 2 * 2 * hv + 2 * hv * d  # projections, gate and beta in, output out (16-bit io)
    weights = C * W * 2 + 8 * hv
    step = 8 * d * d * hv  # one recurrent token: two reductions, the decay and the update
    chunk = hv * (10 * 64 * d + 6 * d * d + 2 * 64 * 64 / 3)  # one token of the chunked form
    log_row = hv * (2 * d + 4) + hk * 2 * d
    op = c["op"]
    if op in ("decode", "verify", "prefill", "layer"):
        state = hv * d * d * (4 if c["state"] == "f32" else 2)
    if op == "decode":
        b = c["batch"]
        return {"bytes": b * (2 * state + 2 * window + token) + weights, "flops": b * step}
    if op == "verify":
        b, t = c["batch"], c["drafts"]
        return {"bytes": b * ((1 + t) * (state + window) + t * token) + weights, "flops": b * t * step}
    if op in ("prefill", "layer"):
        lens, page = _lengths(c), c["page"]
        hits = round(c["hits"] * len(lens))
        states = hits + sum(-(-k // page) for k in lens)
        n = {"bytes": c["tokens"] * token + states * (state + window) + weights, "flops": c["tokens"] * chunk}
        if op == "layer":
            wide = 2 * C + 2 * 2 * hv  # the projections stay inside the layer
            gemm = HIDDEN * (C + 2 * hv * d + 2 * hv)
            n["bytes"] += 2 * gemm + c["tokens"] * (2 * 2 * HIDDEN - wide - 2 * hv * d)
            n["flops"] += 2 * c["tokens"] * gemm
        return n
    ls_state = hv * d * d * 2
    if op == "ls_decode":
        b = c["batch"]
        # a step replays 7.5 logged rows and writes the state every 16th time on average
        return {"bytes": b * (ls_state * 17 / 16 + 8.5 * log_row + 3 * window + token) + weights,
                "flops": b * (step + 7.5 * 2 * d * d * hv)}
    if op == "ls_prefill":
        lens = _lengths(c)
        snaps = sum(-(-k // LS_GRAN) for k in lens)
        ends = sum(2 + (k >= LS_PAGE) for k in lens)
        return {"bytes": c["tokens"] * (token + log_row) + ends * ls_state + snaps * window + weights,
                "flops": c["tokens"] * chunk}
    n, k = c["chains"], c["logged"]
    return {"bytes": n * (2 * ls_state + k * log_row), "flops": n * k * 2 * d * d * hv}


def tolerance(c):
    """Relative 2-norm per output.  A 16-bit output that differs by single
    roundings shows about 2e-3 (bf16) or 3e-4 (f16) against the unrounded
    value; the prefill's f16 matrix operands put about 3e-4 into its fp32
    states; the layer's three roundings in a row show 2.3e-3.  Four times the
    largest output of each case."""
    if c["op"] in ("decode", "verify", "prefill") and c["io"] == "f16":
        return {"rel": 1.6e-3}
    return {"rel": 1e-2 if c["op"] == "layer" else 7e-3}


# ------------------------------------------------------------------ exact (float64)

def _silu(x):
    return x / (1.0 + torch.exp(-x))


def _norm(x):
    return x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def _gates(s, rows=slice(None)):
    g = -torch.exp(s.A_log.double()) * torch.nn.functional.softplus(s.gate[rows].double() + s.dt_bias.double(),
                                                                    threshold=50.0)
    return g, torch.sigmoid(s.beta[rows].double())


def _split(y, c):
    hk, hv, d = c["heads_k"], c["heads_v"], c["dim"]
    q, k, v = y.split([hk * d, hk * d, hv * d], -1)
    return q.unflatten(-1, (hk, d)), k.unflatten(-1, (hk, d)), v.unflatten(-1, (hv, d))


def _conv_step(c, s, x, window, round_conv):
    """SiLU(conv) of one token per sequence in the io dtype's values, and the shifted window."""
    full = torch.cat([window, x[:, :, None]], -1)
    acc = (full.double() * s.weight.double().view(1, -1, W)).sum(-1)
    if round_conv:
        acc = acc.to(x.dtype).double()
    return _silu(acc).to(x.dtype).double(), full[:, :, 1:]


def _recur(c, s, y, g, b, state):
    """One recurrent token: (output, new state, v' rows, normalised k)."""
    r = c["heads_v"] // c["heads_k"]
    q, k, v = _split(y, c)
    q = _norm(q).repeat_interleave(r, 1) * c["dim"] ** -0.5
    kn = _norm(k)
    k = kn.repeat_interleave(r, 1)
    state = state * torch.exp(g)[..., None, None]
    delta = (v - (state * k[..., None]).sum(-2)) * b[..., None]
    state = state + k[..., None] * delta[..., None, :]
    return (state * q[..., None]).sum(-2), state, delta, kn


def _chunked(c, q, k, v, g, b, lens, init, on_end=None):
    """The delta rule in 64-token chunks, all sequences and heads at once
    (sequences that have ended drop out).  q, k, v [T, heads, d], g, b [T,
    HV], init [N, HV, d, d].  Returns (out, v', final states); ``on_end(c,
    sequences, states)`` sees the states after every chunk."""
    d, hv = c["dim"], c["heads_v"]
    r = hv // c["heads_k"]
    T = q.shape[0]
    start = torch.tensor(np.concatenate([[0], np.cumsum(lens)[:-1]]), device=DEV)
    size = torch.tensor(lens, device=DEV)
    out = torch.empty(T, hv, d, device=DEV, dtype=torch.float64)
    vnew = torch.empty_like(out)
    state = init.clone()
    lower = torch.ones(64, 64, device=DEV, dtype=torch.float64).tril(-1)
    for ci in range(-(-max(lens) // 64)):
        live = torch.tensor([i for i, n in enumerate(lens) if n > 64 * ci], device=DEV)
        t = 64 * ci + torch.arange(64, device=DEV)[None]
        ok = t < size[live][:, None]
        rows = torch.where(ok, start[live][:, None] + t, 0)
        m = ok[:, None, :].double()

        def take(x):  # [A, heads, 64, d]
            return x[rows].transpose(1, 2).contiguous()

        kc = take(k).repeat_interleave(r, 1) * m[..., None]
        qc = take(q).repeat_interleave(r, 1) * m[..., None]
        vc = take(v) * m[..., None]
        G = torch.cumsum(take(g[..., None])[..., 0] * m, -1)
        bc = take(b[..., None])[..., 0] * m
        decay = torch.exp((G[..., :, None] - G[..., None, :]).tril()).tril()
        kt = kc.transpose(-1, -2).contiguous()
        L = bc[..., None] * torch.matmul(kc, kt) * decay * lower
        S = state[live]
        eg = torch.exp(G)[..., None]
        vn = bc[..., None] * (vc - eg * torch.matmul(kc, S))
        for i in range(4):  # (I + L) v' = R by 16-token blocks: each block's inverse as a finite product
            a, e = 16 * i, 16 * i + 16
            if i:
                vn[..., a:e, :] -= torch.matmul(L[..., a:e, :a].contiguous(), vn[..., :a, :].contiguous())
            D = -L[..., a:e, a:e].contiguous()
            x = vn[..., a:e, :].contiguous()
            for _ in range(4):  # (I + D)(I + D^2)(I + D^4)(I + D^8)
                x = x + torch.matmul(D, x)
                D = torch.matmul(D, D)
            vn[..., a:e, :] = x
        M = torch.matmul(qc, kt) * decay
        o = (eg * torch.matmul(qc, S) + torch.matmul(M, vn)) * d ** -0.5
        last = G[..., -1:]
        S = torch.exp(last)[..., None] * S + torch.matmul(kt, torch.exp(last - G)[..., None] * vn)
        state[live] = S
        out[rows[ok]] = o.transpose(1, 2)[ok]
        vnew[rows[ok]] = vn.transpose(1, 2)[ok]
        if on_end is not None:
            on_end(ci, live, S)
    return out, vnew, state


def _exact_conv(c, mixed, weight, lens, hist):
    """Packed conv + SiLU in the io dtype's values: y [T, C]."""
    y = torch.empty_like(mixed)
    w = weight.double().view(-1, W)
    a = 0
    for i, n in enumerate(lens):
        for p in range(0, n, 8192):
            e = min(n, p + 8192)
            before = hist[i].t() if p == 0 else mixed[a + p - 3:a + p]
            x = torch.cat([before, mixed[a + p:a + e]]).double()
            acc = sum(x[j:j + e - p] * w[:, j] for j in range(W))
            y[a + p:a + e] = _silu(acc.to(mixed.dtype).double()).to(mixed.dtype)
        a += n
    return y


def _exact_prefill(c, s, lens, hist, init, on_end=None):
    """(out, v', final states, k in the io dtype's values, g) of the packed prompts."""
    q, k, v = _split(_exact_conv(c, s.mixed, s.weight, lens, hist), c)
    q, k = (_norm(x.double()).to(s.mixed.dtype).double() for x in (q, k))
    g, b = _gates(s)
    out, vnew, final = _chunked(c, q, k, v.double(), g, b, lens, init, on_end)
    return out, vnew, final, k, g


def exact(case, seed):
    c = case
    s = prepare(c, seed)
    return {"decode": _exact_steps, "verify": _exact_steps, "prefill": _exact_pool_prefill, "layer": _exact_layer,
            "ls_decode": _exact_ls_decode, "ls_prefill": _exact_ls_prefill, "ls_restore": _exact_ls_restore}[
                c["op"]](c, s)


def _exact_steps(c, s):
    verify = c["op"] == "verify"
    m = s.batch.linear_attn_metadata
    b, t = c["batch"], c.get("drafts", 1)
    if verify:
        _, base, writes = m.verify_groups[t]
        writes = writes.long()
    else:
        base, writes = m.read_slots, m.write_slots[:, None]
    states, conv = s.pool.recurrent_state.double(), s.pool.conv_state.clone()
    S, win = states[base, 0].clone(), conv[base, 0]
    g, beta = (x.view(b, t, -1) for x in _gates(s))
    x = s.mixed.view(b, t, -1)
    out = torch.empty(b, t, c["heads_v"], c["dim"], device=DEV, dtype=torch.float64)
    for i in range(t):
        y, win = _conv_step(c, s, x[:, i], win, verify)
        out[:, i], S, _, _ = _recur(c, s, y, g[:, i], beta[:, i], S)
        states[writes[:, i], 0] = S
        conv[writes[:, i], 0] = win
    return {"out": out.flatten(0, 1), "states": states, "conv": conv.double()}


def _pool_prefill(c, s, io):
    """Exact prefill through the pool's slots: (out, states, conv windows)."""
    lens, page = _lengths(c), c["page"]
    table = s.ctx.state_table
    conv = s.pool.conv_state.clone()
    states = s.pool.recurrent_state.double()
    cached = [q.cached_len for q in s.batch.reqs]
    hist = torch.zeros(len(lens), _conv_dim(c), W - 1, device=DEV, dtype=io.mixed.dtype)
    init = torch.zeros(len(lens), *states.shape[2:], device=DEV, dtype=torch.float64)
    ends = {}
    a = 0
    for i, (n, k) in enumerate(zip(lens, cached)):
        if k:
            slot = int(table[i, k - 1])
            hist[i], init[i] = conv[slot, 0], states[slot, 0]
        for e in [*range(page, n, page), n]:
            ends[i, -(-e // 64) - 1] = int(table[i, k + e - 1])
            rows = [a + e - 3 + j for j in range(3)]
            conv[int(table[i, k + e - 1]), 0] = torch.stack([io.mixed[p] if p >= a else hist[i, :, p - a + 3]
                                                             for p in rows], -1)
        a += n

    def on_end(ci, live, S):
        for j, i in enumerate(live.tolist()):
            if (i, ci) in ends:
                states[ends[i, ci], 0] = S[j]

    out = _exact_prefill(c, io, lens, hist, init, on_end)[0]
    return out, states, conv.double()


def _exact_pool_prefill(c, s):
    out, states, conv = _pool_prefill(c, s, s)
    return {"out": out, "states": states, "conv": conv}


def _exact_layer(c, s):
    """The projections, the GDN output and the norm output are 16-bit tensors between the layer's parts."""
    net, io = s.net, s.x.dtype
    hv, d = c["heads_v"], c["dim"]

    def linear(x, w):
        return torch.matmul(x.double(), w.double().t().contiguous())

    qkvz = linear(s.x, net.in_proj_qkvz_weight).to(io)
    mixed, z = qkvz.split([_conv_dim(c), hv * d], -1)
    beta, gate = linear(s.x, net.in_proj_ba_weight).to(io).chunk(2, -1)
    inner = SimpleNamespace(mixed=mixed.contiguous(), gate=gate, beta=beta, weight=net.conv1d_weight,
                            A_log=net.A_log, dt_bias=net.dt_bias)
    core, states, conv = _pool_prefill(c, s, inner)
    x = core.to(io).double()
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * net.norm.weight.double() * _silu(
        z.reshape(-1, hv, d).double())
    return {"out": linear(y.to(io).flatten(1), net.out_proj_weight), "states": states, "conv": conv}


def _state_index(c, pool, slots):
    """Element indices [slots, HV, d d] of whole states (each head inside one frame) in the states span."""
    hv, d = c["heads_v"], c["dim"]
    byte = torch.arange(hv, device=DEV) * pool.head_payload_bytes
    fr = pool.payload_frame_table[slots.long()][:, byte // LS_FRAME].long()
    at = fr * (LS_FRAME // 2) + (byte % LS_FRAME // 2)
    return at[..., None] + torch.arange(d * d, device=DEV)


def _log_index(c, pool, slots, pos, value):
    """Element indices [rows, heads, d] of the logged value (or key) rows in the logs span."""
    hk, hv, d = c["heads_k"], c["heads_v"], c["dim"]
    keys = LS_GRAN * hk * d
    slots, pos = slots.long()[:, None, None], pos.long()[:, None, None]
    head = torch.arange(hv if value else hk, device=DEV)[None, :, None]
    elem = pos // LS_GRAN * (keys + LS_GRAN * hv * d) + (keys if value else 0) + (
        head * LS_GRAN + pos % LS_GRAN) * d + torch.arange(d, device=DEV)
    fr = pool.payload_frame_table[slots.expand_as(elem), 2 * elem // LS_FRAME].long()
    first = pool.parts.states.shape[0]
    return (fr - first) * (LS_FRAME // 2) + 2 * elem % LS_FRAME // 2


def _decay_index(c, pool, slots, pos):
    """Element indices [rows, HV] of the logged gates in the decays span."""
    first = pool.parts.states.shape[0] + pool.parts.logs.shape[0]
    rec = pool.decay_frame_table[slots.long()].long()
    at = (rec[:, 0] - first) * (LS_FRAME // 4) + rec[:, 1] * (pool.layout.log_decay_bytes // 4)
    return (at + pos.long() * c["heads_v"])[:, None] + torch.arange(c["heads_v"], device=DEV)


def _exact_ls_decode(c, s):
    p, b, r = s.pool.parts, c["batch"], c["heads_v"] // c["heads_k"]
    pos = s.positions.long()
    ids = torch.arange(b, device=DEV)
    logs, states = ids + b, p.states.double().view(-1)
    d = c["dim"]
    where = _state_index(c, s.pool, ids)
    S = states[where].view(b, -1, d, d)
    total = torch.zeros(b, c["heads_v"], device=DEV, dtype=torch.float64)
    add = torch.zeros_like(S)
    for back in range(1, 16):  # the logged tokens since the last write-back, newest first
        on = (pos % 16 >= back).double()[:, None]
        t = (pos - back).clamp_min(0)
        kk = p.logs.view(-1)[_log_index(c, s.pool, logs, t, False)].double().repeat_interleave(r, 1)
        vv = p.logs.view(-1)[_log_index(c, s.pool, logs, t, True)].double()
        add += (on * torch.exp(total))[..., None, None] * kk[..., None] * vv[..., None, :]
        total += on * p.decays.view(-1)[_decay_index(c, s.pool, logs, t)].double()
    S = torch.exp(total)[..., None, None] * S + add
    works = s.pool.conv_frame_table[:b, 0, 0]
    win = s.pool.read_conv(ids, torch.zeros_like(ids), 0)
    y, new = _conv_step(c, s, s.mixed, win, False)
    g, beta = _gates(s)
    out, S, delta, k = _recur(c, s, y, g, beta, S)
    full = pos % 16 == 15
    states[where[full]] = S[full].flatten(2)
    lrow, drow = p.logs.double().view(-1), p.decays.double().view(-1)
    lrow[_log_index(c, s.pool, logs, pos, True)] = delta
    lrow[_log_index(c, s.pool, logs, pos, False)] = k
    drow[_decay_index(c, s.pool, logs, pos)] = g
    conv = p.conv.clone()
    first = sum(x.shape[0] for x in (p.states, p.logs, p.decays))
    for fr in (works, s.pool.conv_frame_table[logs, pos // LS_GRAN, 0]):
        conv[fr.long() - first, :new[0].numel()] = new.flatten(1)
    return {"out": out, "states": states.view(p.states.shape), "logs": lrow.view(p.logs.shape),
            "decays": drow.view(p.decays.shape), "conv": conv.double()}


def _exact_ls_prefill(c, s):
    p, lens = s.pool.parts, _lengths(c)
    n, d, hv = len(lens), c["dim"], c["heads_v"]
    states = p.states.double().view(-1)
    hist = torch.zeros(n, _conv_dim(c), W - 1, device=DEV, dtype=s.mixed.dtype)
    init = torch.zeros(n, hv, d, d, device=DEV, dtype=torch.float64)
    ids = torch.arange(n, device=DEV)

    def on_end(ci, live, S):
        for j, i in enumerate(live.tolist()):
            if lens[i] >= LS_PAGE and 64 * (ci + 1) == lens[i] // LS_PAGE * LS_PAGE:
                states[_state_index(c, s.pool, ids[i:i + 1] + n)] = S[j:j + 1].flatten(2)

    out, vnew, final, k, g = _exact_prefill(c, s, lens, hist, init, on_end)
    states[_state_index(c, s.pool, ids)] = final.flatten(2)
    pos = s.batch.positions
    m = s.batch.linear_attn_metadata
    lrow, drow = p.logs.double().view(-1), p.decays.double().view(-1)
    lrow[_log_index(c, s.pool, m.log_slots, pos % LS_PAGE, True)] = vnew
    lrow[_log_index(c, s.pool, m.log_slots, pos % LS_PAGE, False)] = k
    drow[_decay_index(c, s.pool, m.log_slots, pos % LS_PAGE)] = g
    # conv snapshots are copies of inputs
    return {"out": out, "states": states.view(p.states.shape), "logs": lrow.view(p.logs.shape),
            "decays": drow.view(p.decays.shape), "conv": None}


def _exact_ls_restore(c, s):
    p, n, d = s.pool.parts, c["chains"], c["dim"]
    r = c["heads_v"] // c["heads_k"]
    states = p.states.double().view(-1)
    ids = torch.arange(n, device=DEV)
    S = states[_state_index(c, s.pool, ids)].view(n, -1, d, d)
    for t in range(c["logged"]):
        at = torch.full((n,), t, device=DEV)
        kk = p.logs.view(-1)[_log_index(c, s.pool, 2 * n + ids, at, False)].double().repeat_interleave(r, 1)
        vv = p.logs.view(-1)[_log_index(c, s.pool, 2 * n + ids, at, True)].double()
        g = p.decays.view(-1)[_decay_index(c, s.pool, 2 * n + ids, at)].double()
        S = torch.exp(g)[..., None, None] * S + kk[..., None] * vv[..., None, :]
    states[_state_index(c, s.pool, n + ids)] = S.flatten(2)
    return {"states": states.view(p.states.shape)}
