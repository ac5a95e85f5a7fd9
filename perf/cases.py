"""The decode path's measured cases: one pass each through the package's public entry points.

A case is a plain dict with a ``kind`` (which part of the path) and its sizes:

  request   one whole request through the per-request API: reserve, prefill, decode, release
  topk      one request's Quest selection and its device union (``quest_selection``)
  select    the batched decoder's Quest selection and union for a batch of requests
  resolve   consecutive decode steps' row resolves of a batch
  attend    group attention over a batch's deduplicated rows
  prompt    one layer's write of a prompt: pool rows, host mirror, page bounds
  layer     consecutive decode steps of one sparse layer: append, select, resolve, gather, attend
  dense     the dense launches of one decoder layer's decode step
  head      greedy tokens of the LM head
"""

from __future__ import annotations

from math import ceil

import torch
from torch.nn import functional as F

from mini_hisparse_amd.batched import BatchedSparseDecode, LayerTablesView
from mini_hisparse_amd.config import CacheConfig
from mini_hisparse_amd.dense import (
    argmax_workspace_bytes, gemm_workspace_bytes, linear_argmax_tiled, prepare_add_rms_norm,
    prepare_linear_swiglu_tiled, prepare_linear_tiled, prepare_rotary_split, tile_gate_up, tile_weight,
)
from mini_hisparse_amd.hybrid import HotConfig, HybridKVCache
from mini_hisparse_amd.model import MiniModel, ModelConfig
from mini_hisparse_amd.row_index import GroupEntries
from mini_hisparse_amd.row_kernels import MappedHost, append_rows, append_tokens, attend_groups, pinned_empty
from mini_hisparse_amd.selection import quest_selection, union_bound

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # the command line's demo: the tiny decoder in float32, page budget 3
        dict(name="request-demo", kind="request", hidden=128, ffn=256, layers=2, heads=4, kv=2, vocab=256, prompt=65,
             decode=3, top=3, page=16, dtype="f32"),
        # the smallest call: one short conversation's selection at the 0.5B shape
        dict(name="topk-one", kind="topk", heads=14, kv=2, dim=64, tokens=1999, top=32, page=16, dtype="bf16",
             sink=True),
        # one layer of the 7B shape, 16 histories of up to 128k tokens
        dict(name="select-7b", kind="select", batch=16, heads=28, kv=4, dim=128, tokens=131072, ragged=1021, top=64,
             page=16, dtype="bf16", sink=True),
        dict(name="resolve-7b", kind="resolve", batch=16, heads=28, kv=4, dim=128, tokens=131072, ragged=1021, top=64,
             page=16, hot=32768, steps=4, alike=0.2, dtype="bf16"),
        # the microbench's attention: 64 q / 8 kv heads, 8 requests
        dict(name="attend-8kv", kind="attend", batch=8, heads=64, kv=8, dim=128, union=1800, entries=382, page=16,
             dtype="bf16"),
        # a 7B-shape layer writing a 16k-token prompt, 15% of its pages resident
        dict(name="prompt-16k", kind="prompt", tokens=16383, within=0, kv=4, dim=128, page=16, resident=0.15,
             dtype="bf16"),
        # decode at the 0.5B shape: 4 histories of 32k tokens, hot rows for one step's union
        dict(name="layer-0.5b", kind="layer", batch=4, heads=14, kv=2, dim=64, tokens=32768, ragged=37, top=32, page=16,
             hot=6752, resident=0.25, steps=4, alike=0.8, shared=False),
        # decode at the 7B shape: 8 histories of 128k tokens (host-link bound)
        dict(name="layer-7b", kind="layer", batch=8, heads=28, kv=4, dim=128, tokens=131072, ragged=1021, top=64,
             page=16, hot=32768, resident=0.15, steps=3, alike=0.7, shared=False),
        # the 32B stress shape: pages resampled every step and shared by all heads
        dict(name="layer-32b", kind="layer", batch=3, heads=40, kv=8, dim=128, tokens=65536, ragged=5, top=64, page=16,
             hot=2048, resident=0.4, steps=4, alike=0.0, shared=True),
        dict(name="dense-0.5b", kind="dense", rows=4, hidden=896, heads=14, kv=2, ffn=4864, dtype="bf16"),
        dict(name="dense-7b", kind="dense", rows=8, hidden=3584, heads=28, kv=4, ffn=18944, dtype="bf16"),
        dict(name="head-7b", kind="head", rows=8, hidden=3584, vocab=152064, dtype="bf16"),
    ]


def _log(rng, low, high):
    """A whole number from low to high, spread over its logarithm."""
    return min(high, max(low, round(low * (high / low) ** rng.random())))


# (query heads, KV heads, head dim) of the configurations the framework is run at
_HEADS = ((14, 2, 64), (28, 4, 128), (40, 8, 128), (64, 8, 128), (4, 2, 32), (8, 8, 64), (16, 1, 128))


def draw(rng):
    kind = rng.choice(("topk", "select", "select", "resolve", "attend", "attend", "prompt", "layer", "layer", "dense",
                       "dense", "head", "request"))
    heads, kv, dim = rng.choice(_HEADS)
    case = dict(kind=kind)
    if kind == "request":
        case.update(hidden=128, ffn=256, layers=2, heads=4, kv=2, vocab=256, prompt=_log(rng, 17, 150),
                    decode=rng.randint(2, 5), top=rng.randint(2, 6), page=16, dtype="f32")
    elif kind == "topk":
        case.update(heads=heads, kv=kv, dim=dim, tokens=_log(rng, 200, 60000), top=rng.choice((4, 16, 32, 64)),
                    page=16, dtype=rng.choice(("bf16", "bf16", "f16", "f32")), sink=rng.random() < 0.7)
    elif kind == "select":
        case.update(batch=rng.randint(1, 16), heads=heads, kv=kv, dim=dim, tokens=_log(rng, 1500, 100000),
                    ragged=rng.randint(0, 60), top=rng.choice((8, 32, 64)), page=16,
                    dtype=rng.choice(("bf16", "bf16", "bf16", "f16", "f32")), sink=rng.random() < 0.8)
    elif kind == "resolve":
        heads, kv, dim = rng.choice(_HEADS[:2])
        case.update(batch=rng.randint(1, 16), heads=heads, kv=kv, dim=dim, tokens=_log(rng, 3000, 130000),
                    ragged=rng.randint(0, 90), top=32, page=16, hot=14016 + 64 * rng.randint(0, 290), steps=2, alike=rng.choice((0.3, 0.5, 0.8)), dtype="bf16")
    elif kind == "attend":
        entries = _log(rng, 3, 400)
        case.update(batch=rng.randint(1, 16 if entries < 200 else 8), heads=heads, kv=kv, dim=dim,
                    union=min(2048, entries * rng.randint(1, 4) + rng.randint(0, 9)), entries=entries, page=16,
                    dtype=rng.choice(("bf16", "bf16", "bf16", "f16", "f32")))
    elif kind == "prompt":
        case.update(tokens=_log(rng, 30, 20000), within=rng.randint(0, 15), kv=kv, dim=dim, page=16,
                    resident=rng.choice((0.15, 0.4, 1.0)), dtype=rng.choice(("bf16", "bf16", "f16", "f32")))
    elif kind == "layer":
        shared = rng.random() < 0.4
        heads, kv, dim = rng.choice(_HEADS[:3])
        top = 64 if shared else rng.choice((16, 32))
        case.update(batch=rng.randint(1, 6), heads=heads, kv=kv, dim=dim, tokens=_log(rng, 3000, 50000),
                    ragged=rng.randint(0, 60), top=top, page=16, hot=2048 if shared else 20544,
                    resident=rng.choice((0.15, 0.25, 0.4)), steps=rng.randint(2, 4), alike=0.0 if shared else 0.8,
                    shared=shared)
    elif kind == "dense":
        hidden, heads, kv, ffn = rng.choice(((896, 14, 2, 4864), (1536, 12, 2, 8960), (2048, 16, 2, 11008),
                                             (3584, 28, 4, 18944), (5120, 40, 8, 13824)))
        case.update(rows=rng.randint(1, 16), hidden=hidden, heads=heads, kv=kv, ffn=ffn,
                    dtype=rng.choice(("bf16", "bf16", "f16")))
    else:
        case.update(rows=rng.randint(1, 16), hidden=rng.choice((896, 1536, 3584)), vocab=_log(rng, 8000, 152064),
                    dtype=rng.choice(("bf16", "bf16", "f16")))
    return case


# -- inputs ----------------------------------------------------------------------------

def _generators(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed), torch.Generator().manual_seed(seed)


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEVICE)


def _config(case, blocks, host_pages):
    return CacheConfig(gpu_pages=blocks, host_pages=host_pages, page_size=case["page"], kv_heads=case["kv"],
                       head_dim=case["dim"], device=DEVICE, dtype=DTYPES[case.get("dtype", "bf16")])


def _lengths(case):
    """Ragged histories: each request shorter than the one before it."""
    return [max(case["page"], case["tokens"] - b * case["ragged"]) for b in range(case["batch"])]


def _scales(cpu, kv, dim):
    """Per KV head, 2% of the key channels eight times as large as the others."""
    scale = torch.ones(kv, dim)
    for k in range(kv):
        scale[k, torch.randperm(dim, generator=cpu)[: max(1, round(0.02 * dim))]] = 8.0
    return scale.to(DEVICE)


def _bounds(gen, cpu, pages, case):
    """Lower and upper page bounds, spread like the extrema of 16 normal keys."""
    dtype = DTYPES[case["dtype"]]
    scale = _scales(cpu, case["kv"], case["dim"])
    shape = (pages, case["kv"], case["dim"])
    return (((0.5 * _randn(gen, *shape) - 1.77).clamp(max=-0.01) * scale).to(dtype),
            ((0.5 * _randn(gen, *shape) + 1.77).clamp(min=0.01) * scale).to(dtype))


def _history(case, seed):
    """The layer's history: K and V pages [B, C, 2, P, Hkv, D] and each step's queries
    [steps, B, Hq, D]; a step's query is `alike` to the steps around it."""
    gen, cpu = _generators(seed)
    B, C = case["batch"], ceil(case["tokens"] / case["page"])
    scale = _scales(cpu, case["kv"], case["dim"])
    kv = torch.empty((B, C, 2, case["page"], case["kv"], case["dim"]), dtype=torch.bfloat16, device=DEVICE)
    for b in range(B):
        kv[b] = (_randn(gen, *kv.shape[1:]) * scale).to(torch.bfloat16)
    a = case["alike"]
    shape = (B, case["heads"], case["dim"])
    base = _randn(gen, *shape)
    q = torch.stack([a * base + (1 - a * a) ** 0.5 * _randn(gen, *shape) for _ in range(case["steps"])])
    return kv, q.to(torch.bfloat16), cpu


def _shared_pages(case, cpu):
    """Per step and request, `top` ascending pages drawn uniformly, the tail page last."""
    pages = []
    for _ in range(case["steps"]):
        rows = []
        for length in _lengths(case):
            count = ceil(length / case["page"])
            k = min(case["top"], count)
            row = torch.sort(torch.randperm(count - 1, generator=cpu)[: k - 1]).values.tolist() + [count - 1]
            rows.append(row + [-1] * (case["top"] - k))
        pages.append(torch.tensor(rows, dtype=torch.int32)[:, None].expand(-1, case["heads"], -1).contiguous())
    return pages


def _entries(case, seed):
    """The attention's inputs: queries, pool, each request's union rows (whole pages: even
    ones one block in a row, odd ones scattered over hot rows, as the resolver leaves them),
    and per KV head the union columns its heads read with their head masks.  A request and
    head has up to `entries` pages, the later ones fewer."""
    gen, cpu = _generators(seed)
    B, P, U, Hkv = case["batch"], case["page"], case["union"], case["kv"]
    g = case["heads"] // Hkv
    dtype = DTYPES[case["dtype"]]
    q = _randn(gen, B, case["heads"], case["dim"]).to(dtype)
    blocks = B * U + 3
    pool = torch.empty((blocks, 2, P, Hkv, case["dim"]), dtype=dtype, device=DEVICE)
    for b in range(0, blocks, 4096):
        part = pool[b : b + 4096]
        part.copy_(_randn(gen, *part.shape))
    order = torch.randperm(blocks, generator=cpu)
    whole, loose = order[: B * ((U + 1) // 2)], order[B * ((U + 1) // 2) : B * U]
    rows = torch.empty((B, U, P), dtype=torch.int64)
    rows[:, 0::2] = (whole[:, None] * P + torch.arange(P)).view(B, -1, P)
    scattered = (loose[:, None] * P + torch.arange(P)).reshape(-1)
    rows[:, 1::2] = scattered[torch.randperm(len(scattered), generator=cpu)].view(B, -1, P)
    E = min(case["entries"], U)
    columns = torch.zeros((B, Hkv, E * P), dtype=torch.int32)
    masks = torch.zeros((B, Hkv, E * P), dtype=torch.int32)
    counts = torch.zeros((B, Hkv), dtype=torch.int32)
    share = min(1.0, 1.15 / g)  # a page is read by little over one head of its group
    for b in range(B):
        for k in range(Hkv):
            n = max(1, E - (b + k) % 7 * E // 40)
            pages = torch.sort(torch.randperm(U, generator=cpu)[:n]).values
            bits = torch.rand((n, g), generator=cpu) < share
            bits[torch.arange(n), torch.randint(0, g, (n,), generator=cpu)] = True
            bits[-1] = True  # the tail page is read by every head
            word = (bits.long() << torch.arange(g)).sum(1).to(torch.int32)
            count = n * P - (b * 5 + 3) % P  # a partial tail page
            columns[b, k, : n * P] = (pages[:, None] * P + torch.arange(P)).view(-1).to(torch.int32)
            masks[b, k, : n * P] = word[:, None].expand(n, P).reshape(-1)
            counts[b, k] = count
    return q, pool, rows.view(B, -1), columns, masks, counts


def _dense_weights(case, seed):
    gen, _ = _generators(seed)
    dtype = DTYPES[case["dtype"]]
    hidden, ffn = case["hidden"], case["ffn"]
    dim = hidden // case["heads"]
    new = lambda *shape: (_randn(gen, *shape) * shape[-1] ** -0.5).to(dtype)  # noqa: E731
    wide = hidden + 2 * case["kv"] * dim
    return dict(
        x=_randn(gen, case["rows"], hidden).to(dtype), attn=_randn(gen, case["rows"], hidden).to(dtype),
        norm1=(1 + 0.1 * _randn(gen, hidden)).to(dtype), norm2=(1 + 0.1 * _randn(gen, hidden)).to(dtype),
        qkv=new(wide, hidden), bias=(0.1 * _randn(gen, wide)).to(dtype), o=new(hidden, hidden),
        gate_up=new(2 * ffn, hidden), down=new(hidden, ffn),
        positions=torch.randint(0, 131072, (case["rows"],), generator=gen, device=DEVICE),
    )


def _head_weights(case, seed):
    """An LM head and hidden rows that each favour one token clearly, as a trained model's do."""
    gen, _ = _generators(seed)
    dtype = DTYPES[case["dtype"]]
    weight = (_randn(gen, case["vocab"], case["hidden"]) * case["hidden"] ** -0.5).to(dtype)
    tokens = torch.randint(0, case["vocab"], (case["rows"],), generator=gen, device=DEVICE)
    x = 8 * weight[tokens].float() + _randn(gen, case["rows"], case["hidden"])
    return weight, x.to(dtype), tokens


def _model(case, seed):
    torch.manual_seed(seed)
    model = MiniModel(ModelConfig(case["vocab"], case["hidden"], case["ffn"], case["layers"], case["heads"], case["kv"]))
    gen = torch.Generator().manual_seed(seed + 1)
    tokens = torch.randint(0, case["vocab"], (case["prompt"] + case["decode"],), generator=gen).tolist()
    return model.eval().to(device=DEVICE, dtype=DTYPES[case["dtype"]]), tokens


# -- states ----------------------------------------------------------------------------

def _decoder(case, config, lengths, **options):
    dec = BatchedSparseDecode(config, case["heads"], case["top"], lengths, keep_sink=case.get("sink", True),
                              device=DEVICE, **options)
    for t in (dec.pages, dec.entry_columns, dec.entry_masks, dec.union_physical):
        t.fill_(-1)  # what a short list does not write
    return dec


def _tables(case, pages, cpu, first_hot):
    """Each request's tables: host pages in a row, a share of the pages (and the tail page)
    resident in the first blocks, an empty hot region in slot order."""
    B, C, P, S = case["batch"], ceil(case["tokens"] / case["page"]), case["page"], case["hot"]
    HB = ceil(S / P)
    tags = torch.full((B, S), -1, dtype=torch.int32, device=DEVICE)
    lru = torch.arange(S, dtype=torch.int16, device=DEVICE).repeat(B, 1)
    tables, at = [], 0
    for b in range(B):
        resident = torch.full((C,), -1, dtype=torch.int32)
        resident[pages[b]] = torch.arange(at, at + len(pages[b]), dtype=torch.int32)
        at += len(pages[b])
        hot = torch.arange(first_hot + b * HB, first_hot + (b + 1) * HB, dtype=torch.int32, device=DEVICE)
        source = torch.arange(b * C, (b + 1) * C, dtype=torch.int32, device=DEVICE)
        tables.append(LayerTablesView(source, resident.to(DEVICE), hot, tags[b], lru[b]))
    return tables, tags, lru


def _resident_pages(case, cpu):
    pages = []
    for length in _lengths(case):
        count = ceil(length / case["page"])
        chosen = torch.randperm(count - 1, generator=cpu)[: round(case.get("resident", 0.3) * count)]
        pages.append(torch.sort(torch.cat((chosen, torch.tensor([count - 1])))).values)
    return pages


def prepare(case, seed):
    kind = case["kind"]
    return dict(case=case, **globals()["_prepare_" + kind](case, seed))


def _prepare_request(case, seed):
    model, tokens = _model(case, seed)
    P, total = case["page"], case["prompt"] + case["decode"]
    bound = min(total, (2 + max(0, case["top"] - 2) * case["heads"]) * P)
    hot = HotConfig(bound)
    blocks = 4 * hot.admission_blocks(P, case["layers"])
    config = CacheConfig(gpu_pages=blocks, host_pages=4096, page_size=P, kv_heads=case["kv"],
                         head_dim=case["hidden"] // case["heads"], device=DEVICE, dtype=DTYPES[case["dtype"]])
    return dict(model=model, tokens=tokens, cache=HybridKVCache(config, hot))


def _prepare_topk(case, seed):
    gen, cpu = _generators(seed)
    q = _randn(gen, case["heads"], case["dim"]).to(DTYPES[case["dtype"]])
    lo, hi = _bounds(gen, cpu, ceil(case["tokens"] / case["page"]), case)
    return dict(q=q, lo=lo, hi=hi)


def _prepare_select(case, seed):
    gen, cpu = _generators(seed)
    lengths = _lengths(case)
    bounds = [_bounds(gen, cpu, ceil(n / case["page"]), case) for n in lengths]
    q = _randn(gen, case["batch"], case["heads"], case["dim"]).to(DTYPES[case["dtype"]])
    return dict(dec=_decoder(case, _config(case, 1, 1), lengths), q=q, lo=[b[0] for b in bounds],
                hi=[b[1] for b in bounds])


def _prepare_resolve(case, seed):
    gen, cpu = _generators(seed)
    lengths = _lengths(case)
    bounds = [_bounds(gen, cpu, ceil(n / case["page"]), case) for n in lengths]
    lo, hi = [b[0] for b in bounds], [b[1] for b in bounds]
    config = _config(case, 1, 1)
    base = _randn(gen, case["batch"], case["heads"], case["dim"])
    decoders = []
    a = case["alike"]
    for _ in range(case["steps"]):
        dec = _decoder(case, config, lengths, split_front=True)
        dec.select((a * base + (1 - a * a) ** 0.5 * _randn(gen, *base.shape)).to(torch.bfloat16), lo, hi)
        decoders.append(dec)
    pages = _resident_pages(case, cpu)
    tables, tags, lru = _tables(case, pages, cpu, sum(map(len, pages)))
    return dict(decoders=decoders, tables=tables, tags=tags, lru=lru,
                stats=torch.zeros(3, dtype=torch.int64, device=DEVICE))


def _prepare_attend(case, seed):
    q, pool, rows, columns, masks, counts = _entries(case, seed)
    entries = GroupEntries(columns.to(DEVICE), masks.to(DEVICE), counts.to(DEVICE), columns.shape[2])
    return dict(q=q, pool=pool, rows=rows.to(DEVICE), entries=entries, config=_config(case, pool.shape[0], 1))


def _prepare_prompt(case, seed):
    gen, cpu = _generators(seed)
    P, Hkv, D = case["page"], case["kv"], case["dim"]
    dtype = DTYPES[case["dtype"]]
    pages = ceil((case["within"] + case["tokens"]) / P)
    scale = _scales(cpu, Hkv, D)
    k = (_randn(gen, case["tokens"], Hkv, D) * scale).to(dtype)
    v = _randn(gen, case["tokens"], Hkv, D).to(dtype)
    slots = torch.full((pages,), -1, dtype=torch.int64)
    chosen = torch.randperm(pages, generator=cpu)[: max(1, round(case["resident"] * pages))]
    slots[chosen] = torch.arange(len(chosen))
    host = pinned_empty((pages, 2, P, Hkv, D), dtype)
    host.zero_()
    pool = torch.zeros((len(chosen), 2, P, Hkv, D), dtype=dtype, device=DEVICE)
    lo = torch.full((pages, Hkv, D), float("inf"), dtype=dtype, device=DEVICE)
    return dict(k=k, v=v, slots=slots.tolist(), host_slots=list(range(pages)), pool=pool, host=host,
                alias=MappedHost(host), lo=lo, hi=torch.full_like(lo, float("-inf")),
                config=_config(case, len(chosen), pages))


def _prepare_layer(case, seed):
    kv, q, cpu = _history(case, seed)
    B, C, P = case["batch"], kv.shape[1], case["page"]
    lengths = _lengths(case)
    pages = _resident_pages(case, cpu)
    residents = sum(map(len, pages))
    blocks = residents + B * ceil(case["hot"] / P)
    pool = torch.zeros((blocks, *kv.shape[2:]), dtype=torch.bfloat16, device=DEVICE)
    tables, tags, lru = _tables(case, pages, cpu, residents)
    lo, hi, device_rows, host_rows, new = [], [], [], [], []
    at = 0
    for b, length in enumerate(lengths):
        pool[at : at + len(pages[b])] = kv[b, pages[b].to(DEVICE)]
        at += len(pages[b])
        tail, off = divmod(length - 1, P)
        lo.append(kv[b, :, 0].amin(1).contiguous())
        hi.append(kv[b, :, 0].amax(1).contiguous())
        lo[b][tail], hi[b][tail] = kv[b, tail, 0, : off + 1].amin(0), kv[b, tail, 0, : off + 1].amax(0)
        device_rows.append((at - 1) * P + off)
        host_rows.append((b * C + tail) * P + off)
        new.append(kv[b, tail, :, off])
    new = torch.stack(new, 1)  # [2, B, Hkv, D]: the newest token's K and V
    host = pinned_empty((B * C, *kv.shape[2:]), torch.bfloat16)
    host.copy_(kv.view(B * C, *kv.shape[2:]))
    tails = [(length - 1) // P for length in lengths]
    return dict(
        dec=_decoder(case, _config(case, blocks, B * C), lengths, shared_selection=case["shared"], split_front=True),
        config=_config(case, blocks, B * C), q=list(q), lo=lo, hi=hi, k=new[0].contiguous(), v=new[1].contiguous(),
        tail_lo=[lo[b][t] for b, t in enumerate(tails)], tail_hi=[hi[b][t] for b, t in enumerate(tails)],
        device_rows=device_rows, host_rows=host_rows, host=host, alias=MappedHost(host), pool=pool, tables=tables,
        tags=tags, lru=lru, stats=torch.zeros(3, dtype=torch.int64, device=DEVICE),
        pages=[p.to(DEVICE) for p in _shared_pages(case, cpu)] if case["shared"] else None,
    )


def _prepare_dense(case, seed):
    w = _dense_weights(case, seed)
    rows, hidden, ffn, heads, kv = (case[n] for n in ("rows", "hidden", "ffn", "heads", "kv"))
    dim = hidden // heads
    new = lambda *shape: torch.empty(shape, dtype=w["x"].dtype, device=DEVICE)  # noqa: E731
    x, h, o, delta, act = new(rows, hidden), new(rows, hidden), new(rows, hidden), new(rows, hidden), new(rows, ffn)
    wide = w["qkv"].shape[0]
    qkv, q, k, v = new(rows, wide), new(rows, heads, dim), new(rows, kv, dim), new(rows, kv, dim)
    tiles = dict(qkv=tile_weight(w["qkv"]), o=tile_weight(w["o"]), down=tile_weight(w["down"]),
                 gate_up=tile_gate_up(w["gate_up"], ffn))
    need = max(gemm_workspace_bytes(rows, n, k_) for n, k_ in ((wide, hidden), (hidden, hidden), (hidden, ffn)))
    ws = torch.empty(need, dtype=torch.uint8, device=DEVICE)
    launches = [  # every argument bound once, as the engine does
        prepare_add_rms_norm(x, None, w["norm1"], 1e-6, h),
        prepare_linear_tiled(h, tiles["qkv"], wide, w["bias"], qkv, ws),
        prepare_rotary_split(qkv, w["positions"], heads, kv, dim, 1e6, (q, k, v)),
        prepare_linear_tiled(w["attn"], tiles["o"], hidden, None, o, ws),
        prepare_add_rms_norm(x, o, w["norm2"], 1e-6, h),
        prepare_linear_swiglu_tiled(h, tiles["gate_up"], ffn, act),
        prepare_linear_tiled(act, tiles["down"], hidden, None, delta, ws),
    ]
    keep = (h, o, act, qkv, ws, w["norm1"], w["norm2"], w["bias"], w["attn"], w["positions"], tiles)
    return dict(launches=launches, x0=w["x"], out=(x, q, k, v, delta), keep=keep)


def _prepare_head(case, seed):
    weight, x, _ = _head_weights(case, seed)
    ws = torch.empty(argmax_workspace_bytes(case["rows"], case["vocab"], case["hidden"]), dtype=torch.uint8, device=DEVICE)
    return dict(x=x, tiles=tile_weight(weight), ws=ws,
                out=torch.empty(case["rows"], dtype=torch.int64, device=DEVICE))


# -- passes ----------------------------------------------------------------------------

def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


def _run_request(s):
    case, model, cache = s["case"], s["model"], s["cache"]
    prompt, rest = s["tokens"][: case["prompt"]], s["tokens"][case["prompt"] :]
    cache.reserve("r", len(s["tokens"]), case["layers"])
    logits = [model.prefill(prompt, cache, "r")]
    for token in rest:
        logits.append(model.decode(token, "r", cache, case["top"]))
    cache.release_request("r")
    return logits


def _run_topk(s):
    case = s["case"]
    selection = quest_selection(s["q"], s["lo"], s["hi"], case["tokens"], case["page"], case["top"], case["sink"])
    topk = selection.logical_topk(s["q"].device)
    return [selection.device_pages, topk.positions, topk.head_columns, topk.union_count, topk.entries.counts]


def _run_select(s):
    dec = s["dec"]
    dec.select(s["q"], s["lo"], s["hi"])
    return [dec.pages, dec.positions, dec.head_columns, dec.union_count, dec.entry_columns, dec.entry_masks,
            dec.entry_counts, dec.status]


def _run_resolve(s):
    for dec in s["decoders"]:
        dec.resolve(s["tables"], row_stats=s["stats"])
    return [t for dec in s["decoders"] for t in (dec.union_physical, dec.row_counts)] + [s["tags"], s["lru"], s["stats"]]


def _run_attend(s):
    return attend_groups(s["q"], s["pool"], s["rows"], s["entries"], s["config"])


def _run_prompt(s):
    case = s["case"]
    append_tokens(s["k"], s["v"], 0, case["within"], s["slots"], s["host_slots"], s["pool"], s["alias"], s["lo"],
                  s["hi"], None, s["config"])
    return [s["pool"], s["host"], s["lo"], s["hi"]]


def _run_layer(s):
    dec, pool, outs = s["dec"], s["pool"], []
    for step, q in enumerate(s["q"]):
        append_rows(s["k"], s["v"], pool, s["device_rows"], s["tail_lo"], s["tail_hi"], s["config"], host=s["alias"],
                    host_rows=s["host_rows"])
        if s["pages"] is None:
            dec.select(q, s["lo"], s["hi"])
        else:
            dec.select_pages(s["pages"][step], validate=False)
        dec.resolve(s["tables"], row_stats=s["stats"])
        dec.gather(s["alias"], pool, None)
        outs.append(dec.attend(q, pool))
    return [outs, s["tags"], s["lru"], dec.row_counts, pool, dec.status]


def _run_dense(s):
    x = s["out"][0]
    x.copy_(s["x0"])
    stream = torch.cuda.current_stream(x.device).cuda_stream
    for launch in s["launches"]:
        launch(stream)
    return list(s["out"])


def _run_head(s):
    return linear_argmax_tiled(s["x"], s["tiles"], s["case"]["vocab"], None, out=s["out"], workspace=s["ws"])


# -- the same in 64 bits ---------------------------------------------------------------------

def exact(case, seed):
    kind = case["kind"]
    if kind == "request":
        return _exact_request(case, seed)
    if kind == "attend":
        return _exact_attend(case, seed)
    if kind == "layer":
        return _exact_layer(case, seed)
    if kind == "dense":
        return _exact_dense(case, seed)
    return None  # whole numbers, and rows copied as they are


def _page_choice(q, lo, hi, count, top, sink=True):
    """The chosen pages [H, min(top, count)]: scores summed over the channels in ascending
    order in float32 (the order that decides near ties), ties to the lower page."""
    if top >= count:
        return torch.arange(count, device=q.device).expand(q.shape[0], count)
    g = q.shape[0] // lo.shape[1]
    lo, hi, q = lo[:count].float(), hi[:count].float(), q.float()
    scores = torch.zeros((q.shape[0], count), device=q.device)
    for d in range(q.shape[1]):
        column = q[:, d : d + 1]
        bound = torch.where(column >= 0, hi[:, :, d].T.repeat_interleave(g, 0), lo[:, :, d].T.repeat_interleave(g, 0))
        scores = scores + column * bound
    scores[:, count - 1] = float("inf")
    if sink and top > 1:
        scores[:, 0] = float("inf")
    return scores.sort(descending=True, stable=True).indices[:, :top].sort().values


def _paged_attention(q, kv, pages, length):
    """Attention of q [H, D] over each head's pages [H, k] of kv [C, 2, P, Hkv, D], in float64."""
    H, D = q.shape
    P, Hkv = kv.shape[2], kv.shape[3]
    head = torch.arange(H, device=q.device) // (H // Hkv)
    rows = kv.permute(3, 0, 1, 2, 4)[head[:, None], pages].double()  # [H, k, 2, P, D]
    scores = torch.einsum("hd,hkpd->hkp", q.double(), rows[:, :, 0]) * D**-0.5
    token = pages[:, :, None] * P + torch.arange(P, device=q.device)
    weights = scores.masked_fill(token >= length, float("-inf")).flatten(1).softmax(-1)
    return (weights[:, :, None] * rows[:, :, 1].flatten(1, 2)).sum(1)


def _exact_request(case, seed):
    model, tokens = _model(case, seed)
    model = model.double()
    cfg, P = model.config, case["page"]
    T, D = len(tokens), cfg.head_dim
    H, Hkv = cfg.num_attention_heads, cfg.num_key_value_heads
    x = model.model.embed_tokens.weight[torch.tensor(tokens, device=DEVICE)]
    inverse = cfg.rope_theta ** (-torch.arange(0, D, 2, device=DEVICE).float() / D)
    angle = (torch.arange(T, device=DEVICE).float()[:, None] * inverse).double()
    cos, sin = torch.cat((angle, angle), -1).cos()[:, None], torch.cat((angle, angle), -1).sin()[:, None]

    def norm(t, weight):
        return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + cfg.rms_norm_eps) * weight

    def turn(t):
        a, b = t.chunk(2, -1)
        return t * cos + torch.cat((-b, a), -1) * sin

    with torch.no_grad():
        for layer in model.model.layers:
            attn, mlp = layer.self_attn, layer.mlp
            h = norm(x, layer.input_layernorm.weight)
            q, k = turn(attn.q_proj(h).view(T, H, D)), turn(attn.k_proj(h).view(T, Hkv, D))
            v = attn.v_proj(h).view(T, Hkv, D)
            out = []
            for t in range(T):
                n = t + 1
                pages = ceil(n / P)
                kv = torch.zeros((pages * P, 2, Hkv, D), dtype=torch.float64, device=DEVICE)
                kv[:n, 0], kv[:n, 1] = k[:n], v[:n]
                kv = kv.view(pages, P, 2, Hkv, D).transpose(1, 2)
                if t < case["prompt"]:
                    chosen = torch.arange(pages, device=DEVICE).expand(H, pages)
                else:
                    keys = torch.full((pages * P, Hkv, D), float("nan"), dtype=torch.float64, device=DEVICE)
                    keys[:n] = k[:n]
                    keys = keys.view(pages, P, Hkv, D)
                    lo = keys.nan_to_num(float("inf")).amin(1)
                    hi = keys.nan_to_num(float("-inf")).amax(1)
                    chosen = _page_choice(q[t], lo, hi, pages, case["top"])
                out.append(_paged_attention(q[t], kv, chosen, n))
            x = x + attn.o_proj(torch.stack(out).view(T, -1))
            h = norm(x, layer.post_attention_layernorm.weight)
            x = x + mlp.down_proj(F.silu(mlp.gate_proj(h)) * mlp.up_proj(h))
        logits = model.lm_head(norm(x, model.model.norm.weight))
    return [logits[t] for t in range(case["prompt"] - 1, T)]


def _exact_attend(case, seed):
    q, pool, rows, columns, masks, counts = _entries(case, seed)
    B, Hkv, D, P = case["batch"], case["kv"], case["dim"], case["page"]
    g = case["heads"] // Hkv
    out = torch.zeros((B, case["heads"], D), dtype=torch.float64, device=DEVICE)
    for b in range(B):
        for k in range(Hkv):
            n = int(counts[b, k])
            at = rows[b][columns[b, k, :n].long()].to(DEVICE)
            K, V = (pool[at // P, plane, at % P, k].double() for plane in (0, 1))
            query = q[b, k * g : (k + 1) * g].double()
            read = (masks[b, k, :n].to(DEVICE)[None] >> torch.arange(g, device=DEVICE)[:, None]) & 1
            scores = (query @ K.T * D**-0.5).masked_fill(read == 0, float("-inf"))
            out[b, k * g : (k + 1) * g] = scores.softmax(-1) @ V
    return out


def _exact_layer(case, seed):
    kv, q, cpu = _history(case, seed)
    lengths = _lengths(case)
    _resident_pages(case, cpu)
    shared = _shared_pages(case, cpu) if case["shared"] else None
    P, outs = case["page"], [torch.empty(q.shape[1:], dtype=torch.float64, device=DEVICE) for _ in q]
    for b, length in enumerate(lengths):
        count = ceil(length / P)
        off = length - (count - 1) * P
        lo, hi = kv[b, :, 0].amin(1), kv[b, :, 0].amax(1)
        lo[count - 1], hi[count - 1] = kv[b, count - 1, 0, :off].amin(0), kv[b, count - 1, 0, :off].amax(0)
        for step, query in enumerate(q):
            if shared is None:
                pages = _page_choice(query[b], lo, hi, count, case["top"])
            else:
                pages = shared[step][b, :, : min(case["top"], count)].long().to(DEVICE)
            outs[step][b] = _paged_attention(query[b], kv[b], pages, length)
    return [outs, None, None, None, None, None]


def _exact_dense(case, seed):
    w = {name: t if name == "positions" else t.double() for name, t in _dense_weights(case, seed).items()}
    rows, heads, kv = case["rows"], case["heads"], case["kv"]
    dim = case["hidden"] // heads

    def norm(t, weight):
        return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + 1e-6) * weight

    def turn(t):
        inverse = 1e6 ** (-torch.arange(0, dim, 2, device=DEVICE).float() / dim)
        angle = (w["positions"].float()[:, None] * inverse).double()
        cos, sin = torch.cat((angle, angle), -1).cos()[:, None], torch.cat((angle, angle), -1).sin()[:, None]
        a, b = t.chunk(2, -1)
        return t * cos + torch.cat((-b, a), -1) * sin

    qkv = norm(w["x"], w["norm1"]) @ w["qkv"].T + w["bias"]
    q, k, v = (t.reshape(rows, -1, dim) for t in qkv.split([heads * dim, kv * dim, kv * dim], 1))
    x = w["x"] + w["attn"] @ w["o"].T
    gate, up = (norm(x, w["norm2"]) @ w["gate_up"].T).chunk(2, 1)
    return [x, turn(q), turn(k), v, (F.silu(gate) * up) @ w["down"].T]


# -- what a pass cannot do without ---------------------------------------------------------------

def work(case):
    kind = case["kind"]
    size = DTYPES[case.get("dtype", "bf16")].itemsize
    if kind == "request":
        layer = 2 * case["hidden"] ** 2 + 2 * case["hidden"] * (case["hidden"] // case["heads"]) * case["kv"] + \
            3 * case["hidden"] * case["ffn"]
        weights = case["layers"] * layer + case["hidden"] * case["vocab"]
        passes = 1 + case["decode"]
        return {"bytes": weights * size * passes, "flops": 2 * weights * (case["prompt"] + case["decode"])}
    if kind == "topk":
        pages = ceil(case["tokens"] / case["page"])
        return _select_work(case, [case["tokens"]], size, pages)
    if kind == "select":
        return _select_work(case, _lengths(case), size, sum(ceil(n / case["page"]) for n in _lengths(case)))
    if kind == "resolve":
        return {"bytes": case["steps"] * _resolve_bytes(case), "flops": 0}
    if kind == "attend":
        rows = 0
        E = min(case["entries"], case["union"])
        for b in range(case["batch"]):
            for k in range(case["kv"]):
                rows += max(1, E - (b + k) % 7 * E // 40) * case["page"] - (b * 5 + 3) % case["page"]
        heads = case["batch"] * case["heads"]
        g = case["heads"] // case["kv"]
        return {"bytes": rows * (2 * case["dim"] * size + 16) + 2 * heads * case["dim"] * size,
                "flops": 4 * rows * g * case["dim"]}
    if kind == "prompt":
        row = 2 * case["kv"] * case["dim"] * size
        return {"bytes": case["tokens"] * row * (2 + case["resident"]) + 2 * ceil(case["tokens"] / 16) * row, "flops": 0}
    if kind == "layer":
        row = 2 * case["kv"] * case["dim"] * 2
        heads = 1 if case["shared"] else case["heads"] // case["kv"]
        total, flops = 0, 0
        for n in _lengths(case):
            read = union_bound(n, case["page"], case["top"], heads, True)
            total += read * row
            flops += 4 * read * case["heads"] * case["dim"]
        if not case["shared"]:
            chosen = _select_work(case, _lengths(case), 2, sum(ceil(n / case["page"]) for n in _lengths(case)))
            total, flops = total + chosen["bytes"], flops + chosen["flops"]
        return {"bytes": case["steps"] * (total + _resolve_bytes(case)), "flops": case["steps"] * flops}
    if kind == "dense":
        dim = case["hidden"] // case["heads"]
        weights = case["hidden"] * (2 * case["hidden"] + 2 * case["kv"] * dim + 3 * case["ffn"])
        return {"bytes": weights * size + 8 * case["rows"] * case["hidden"] * size, "flops": 2 * weights * case["rows"]}
    weights = case["hidden"] * case["vocab"]
    return {"bytes": weights * size, "flops": 2 * weights * case["rows"]}


def _select_work(case, lengths, size, pages):
    """Page bounds and queries read; pages and each head's columns written."""
    width = sum(min(case["top"] * case["page"], n) for n in lengths)
    return {"bytes": 2 * pages * case["kv"] * case["dim"] * size + len(lengths) * case["heads"] * case["dim"] * size +
            4 * len(lengths) * case["heads"] * case["top"] + 8 * case["heads"] * width,
            "flops": 3 * pages * case["heads"] * case["dim"]}


def _resolve_bytes(case):
    """Tags, LRU and page tables read, tags and LRU written, each selected row's token and place."""
    heads = 1 if case.get("shared") else case["heads"]
    rows = sum(union_bound(n, case["page"], case["top"], heads, True) for n in _lengths(case))
    return case["batch"] * case["hot"] * 12 + sum(8 * ceil(n / case["page"]) for n in _lengths(case)) + 12 * rows


def tolerance(case):
    """About four times what was seen between summation orders (attention splits dealt or in
    chunks; the projections against PyTorch's), or against 64 bits for float32."""
    kind = case["kind"]
    if kind in ("request", "attend", "layer", "dense"):
        return {"f32": {"rel": 1.5e-6, "max": 1.5e-5}, "f16": {"rel": 1e-3, "max": 1.2e-2},
                "bf16": {"rel": 6e-3, "max": 5e-2}}[case.get("dtype", "bf16")]
    return "exact"
