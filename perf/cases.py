"""Workloads of the paged-KV path: what is timed when the framework's speed is compared.

Every case is one call (or one whole loop-step) of the public entry points at
the shapes of this repository's own workloads: 16 query / 16 KV heads x 128,
pages of 16 tokens, bf16, over the context ranges of its benchmark, plus the
other storage types and the grouped-query heads that its tests cover.

A case holds plain sizes.  Its context lengths are a fixed spread over
[lo, hi] (so the work of a case is known without a seed); the seed draws the
data, the page permutation, the order of the rows and their loop depths.
"""

from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parent.parent / "vllm-rlt_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from vllm_rlt_amd import ops  # noqa: E402
from vllm_rlt_amd.paged_attention import HipPagedAttention  # noqa: E402

PAGE = 16
LOOPS = 4
LAYERS = 24
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEVICE = "cuda"


def listed():
    return [
        # A handful of short requests, one layer: the smallest decode call, all latency.
        dict(name="decode-few", kind="decode", rows=4, lo=1, hi=256, hq=16, hkv=16, d=128, dtype="bf16", planes=4),
        # The everyday serving batch: 64 requests at mixed loop depths, one storage plane per depth.
        dict(name="decode-last-exited", kind="decode", rows=64, lo=512, hi=4096, hq=16, hkv=16, d=128, dtype="bf16", planes=4),
        # A full batch of longer requests on the one-plane layout: the largest decode call.
        dict(name="decode-shared", kind="decode", rows=256, lo=1024, hi=8192, hq=16, hkv=16, d=128, dtype="bf16", planes=1),
        # Two users with long documents: few rows, each of many splits.
        dict(name="decode-long", kind="decode", rows=2, lo=16384, hi=32768, hq=16, hkv=16, d=128, dtype="bf16", planes=1),
        # A grouped-query model in fp16 at a medium batch.
        dict(name="decode-gqa", kind="decode", rows=24, lo=512, hi=4096, hq=32, hkv=8, d=128, dtype="fp16", planes=1),
        # Requests that share a cached system prompt, per loop depth one aliased prefix.
        dict(name="decode-prefix", kind="prefix", rows=64, lo=4096, hi=8192, prefix=2048, hq=16, hkv=16, d=128, dtype="bf16", planes=4),
        # Chunked prefill under load: eight 512-token chunks over their paged prefixes.
        dict(name="prefill-chunks", kind="prefill", seqs=8, clo=512, chi=512, lo=0, hi=16384, hq=16, hkv=16, d=128, dtype="bf16"),
        # New requests of ordinary, ragged prompt lengths, some over a cached prefix.
        dict(name="prefill-ragged", kind="prefill", seqs=6, clo=9, chi=331, lo=0, hi=2048, hq=16, hkv=16, d=128, dtype="bf16"),
        # One user's long document: a chunk at the end of a long prefix, nothing else to run beside it.
        dict(name="prefill-long", kind="prefill", seqs=1, clo=512, chi=512, lo=16000, hi=16000, hq=16, hkv=16, d=128, dtype="bf16"),
        # The 32-bit storage type, used to check a model against its reference.
        dict(name="prefill-fp32", kind="prefill", seqs=3, clo=61, chi=200, lo=0, hi=700, hq=16, hkv=16, d=128, dtype="fp32"),
        # The rotation and KV write of a packed prefill chunk, before its attention.
        dict(name="rope-append", kind="rope", rows=4096, hq=16, hkv=16, d=128, dtype="bf16"),
        # A whole recurrent pass of a small interactive batch: routing metadata, 24 layers, exit copies.
        dict(name="loop-step", kind="step", rows=8, lo=64, hi=1024, hq=16, hkv=16, d=128, dtype="bf16", planes=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges: any batch, raggedness, storage type and head grouping between them."""
    kind = rng.choices(["decode", "prefix", "prefill", "prefill-fp32", "rope", "step"], weights=[6, 1, 5, 1, 1, 1])[0]
    hq, hkv = rng.choice([(16, 16), (16, 16), (16, 16), (32, 8)])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    if kind == "decode":
        rows = _log(rng, 1, 256)
        cap = min(32768, 256 * 8192 // 2 // rows)
        hi = _log(rng, 100, cap)
        return dict(kind="decode", rows=rows, lo=rng.randint(1, hi), hi=hi, hq=hq, hkv=hkv, d=128, dtype=dtype,
                    planes=rng.choice([1, 4]) if rows * hi <= 64 * 4096 else 1)
    if kind == "prefix":
        hi = _log(rng, 4096, 8192)
        return dict(kind="prefix", rows=rng.randint(8, 64), lo=rng.randint(2200, hi), hi=hi, prefix=PAGE * rng.randint(32, 128),
                    hq=16, hkv=16, d=128, dtype="bf16", planes=rng.choice([1, 4]))
    if kind == "prefill":
        seqs = _log(rng, 1, 24)
        chi = _log(rng, 5, min(1024, 4096 // seqs))
        return dict(kind="prefill", seqs=seqs, clo=rng.randint(1, chi), chi=chi, lo=0, hi=_log(rng, 16, 16384), hq=hq, hkv=hkv,
                    d=128, dtype=dtype)
    if kind == "prefill-fp32":
        chi = _log(rng, 5, 200)
        return dict(kind="prefill", seqs=rng.randint(1, 3), clo=rng.randint(1, chi), chi=chi, lo=0, hi=_log(rng, 16, 700), hq=16,
                    hkv=16, d=128, dtype="fp32")
    if kind == "rope":
        return dict(kind="rope", rows=_log(rng, 1, 4096), hq=hq, hkv=hkv, d=128, dtype=dtype)
    hi = _log(rng, 64, 1024)
    return dict(kind="step", rows=rng.randint(1, 8), lo=rng.randint(1, hi), hi=hi, hq=16, hkv=16, d=128, dtype="bf16", planes=4)


# ------------------------------------------------------------------ lengths
def _spread(n, lo, hi):
    """n lengths evenly over [lo, hi]: the same ones for every seed."""
    return [lo + int((hi - lo) * (i + 0.5) / n) for i in range(n)]


def _contexts(case):
    return _spread(case["rows"], case["lo"], case["hi"])


def _chunks(case):
    """(prefix, chunk) of each sequence: both spread evenly, paired by a fixed shuffle."""
    n = case["seqs"]
    chunks = _spread(n, case["clo"], case["chi"])
    random.Random(n).shuffle(chunks)
    return list(zip(_spread(n, case["lo"], case["hi"]), chunks))


def _depths(case):
    return [i % LOOPS for i in range(case["rows"])]


def _exits(case):
    """(row, exit depth) of a loop-step's tokens that stop before the last loop."""
    return [(r, d) for r, d in enumerate(_depths(case)) if d < LOOPS - 1 and r % 2 == 0]


def _esize(case):
    return 4 if case["dtype"] == "fp32" else 2


# ------------------------------------------------------------------- inputs
def _pages(tokens):
    return -(-tokens // PAGE)


def _pool(gen, blocks, layers, case):
    shape = (blocks, layers, PAGE, case["hkv"], case["d"])
    dtype = DTYPES[case["dtype"]]
    return [torch.empty(shape, dtype=dtype, device=DEVICE).normal_(generator=gen) for _ in range(2)]


def _normal(gen, *shape, dtype):
    return torch.empty(shape, dtype=dtype, device=DEVICE).normal_(generator=gen)


def _tables(host, lengths, planes, prefix_pages=0):
    """int32 [rows, planes, width] tables of random pages; the first prefix_pages of a plane are the same in every row."""
    need = [_pages(n) for n in lengths]
    blocks = planes * (prefix_pages + sum(n - prefix_pages for n in need))
    perm = torch.randperm(blocks, generator=host, dtype=torch.int64).to(torch.int32)
    tables = torch.zeros(len(lengths), planes, max(need), dtype=torch.int32)
    shared = perm[: planes * prefix_pages].view(planes, prefix_pages)
    at = planes * prefix_pages
    for r, n in enumerate(need):
        own = n - prefix_pages
        for p in range(planes):
            tables[r, p, :prefix_pages] = shared[p]
            tables[r, p, prefix_pages:n] = perm[at : at + own]
            at += own
    return tables, blocks, shared


def prepare(case, seed):
    host = torch.Generator().manual_seed(seed)
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    return _PREPARE[case["kind"]](case, host, gen)


def _prepare_decode(case, host, gen):
    rows, planes, dtype = case["rows"], case["planes"], DTYPES[case["dtype"]]
    order = torch.randperm(rows, generator=host).tolist()
    contexts = _contexts(case)
    lengths = [contexts[i] + 1 for i in order]  # the new token is part of the context
    prefix_pages = case.get("prefix", 0) // PAGE
    tables, blocks, shared = _tables(host, lengths, planes, prefix_pages)
    depths = [_depths(case)[i] % planes for i in order]
    mine = tables[torch.arange(rows), torch.tensor(depths)].contiguous()
    last = torch.tensor(lengths) - 1
    key, value = _pool(gen, blocks, 1, case)
    state = dict(
        case=case, lengths=lengths, key=key, value=value, tables=mine.to(DEVICE),
        context_lengths=torch.tensor(lengths, dtype=torch.int32, device=DEVICE),
        blocks=mine[torch.arange(rows), last // PAGE].long().to(DEVICE), offsets=(last % PAGE).to(DEVICE),
        q=_normal(gen, rows, case["hq"], case["d"], dtype=dtype), k=_normal(gen, rows, case["hkv"], case["d"], dtype=dtype),
        v=_normal(gen, rows, case["hkv"], case["d"], dtype=dtype),
        attention=HipPagedAttention(DEVICE, dtype, case["d"], PAGE), groups=None,
    )
    if prefix_pages:
        pages = [shared[d].tolist() for d in depths]
        state["groups"] = ops.prefix_groups(pages, lengths, PAGE, case["hq"] // case["hkv"], DEVICE)
    return state


def _prepare_prefill(case, host, gen):
    dtype = DTYPES[case["dtype"]]
    pairs = _chunks(case)
    pairs = [pairs[i] for i in torch.randperm(len(pairs), generator=host).tolist()]
    lengths = [p + c for p, c in pairs]
    tables, blocks, _ = _tables(host, lengths, 1)
    chunks = [c for _, c in pairs]
    cu = [0]
    for c in chunks:
        cu.append(cu[-1] + c)
    key, value = _pool(gen, blocks, 1, case)
    return dict(
        case=case, lengths=lengths, chunks=chunks, key=key, value=value, tables=tables[:, 0].contiguous().to(DEVICE),
        context_lengths=torch.tensor(lengths, dtype=torch.int32, device=DEVICE),
        cu=torch.tensor(cu, dtype=torch.int32, device=DEVICE), q=_normal(gen, cu[-1], case["hq"], case["d"], dtype=dtype),
        attention=HipPagedAttention(DEVICE, dtype, case["d"], PAGE),
    )


def _prepare_rope(case, host, gen):
    rows, d, dtype = case["rows"], case["d"], DTYPES[case["dtype"]]
    # A packed chunk writes whole runs of consecutive slots, page after random page.
    blocks = _pages(rows) + 8
    perm = torch.randperm(blocks, generator=host)
    t = torch.arange(rows)
    key, value = _pool(gen, blocks, 1, case)
    inverse = 1.0 / (1e6 ** (torch.arange(0, d, 2, device=DEVICE).float() / d))
    start = int(torch.randint(0, 4096, (1,), generator=host))
    angle = torch.cat([torch.outer(torch.arange(rows, device=DEVICE).float() + start, inverse)] * 2, dim=-1)
    return dict(
        case=case, key=key, value=value, blocks=perm[t // PAGE].to(DEVICE), offsets=(t % PAGE).to(DEVICE),
        q=_normal(gen, rows, case["hq"], d, dtype=dtype), k=_normal(gen, rows, case["hkv"], d, dtype=dtype),
        v=_normal(gen, rows, case["hkv"], d, dtype=dtype), cos=angle.cos().to(dtype), sin=angle.sin().to(dtype),
    )


def _prepare_step(case, host, gen):
    rows, planes, dtype = case["rows"], case["planes"], DTYPES[case["dtype"]]
    order = torch.randperm(rows, generator=host).tolist()
    contexts = _contexts(case)
    # Row r of the batch is request slot order[r]; its new token is at position contexts[slot].
    tables, blocks, _ = _tables(host, [n + 1 for n in contexts], planes)
    depths = _depths(case)
    descriptors = torch.tensor([[s, depths[s], contexts[s]] for s in order], dtype=torch.int64)
    exits = torch.tensor([[s, d, contexts[s]] for s, d in _exits(case)], dtype=torch.int64).view(-1, 3)
    key, value = _pool(gen, blocks, LAYERS, case)
    width = tables.shape[2]

    def i64(n):
        return torch.zeros(n, dtype=torch.int64, device=DEVICE)

    attention = HipPagedAttention(DEVICE, dtype, case["d"], PAGE)
    return dict(
        case=case, order=order, key=key, value=value, tables=tables.to(DEVICE), descriptors=descriptors.to(DEVICE),
        exits=exits.to(DEVICE), slots=i64(rows), positions=i64(rows), blocks=i64(rows), offsets=i64(rows),
        lengths=torch.zeros(rows, dtype=torch.int32, device=DEVICE),
        row_tables=torch.zeros(rows, width, dtype=torch.int32, device=DEVICE), width=width,
        q=[_normal(gen, rows, case["hq"], case["d"], dtype=dtype) for _ in range(LAYERS)],
        k=[_normal(gen, rows, case["hkv"], case["d"], dtype=dtype) for _ in range(LAYERS)],
        v=[_normal(gen, rows, case["hkv"], case["d"], dtype=dtype) for _ in range(LAYERS)], attention=attention,
        layers=[(key[:, i], value[:, i]) for i in range(LAYERS)],
    )


_PREPARE = {
    "decode": _prepare_decode, "prefix": _prepare_decode, "prefill": _prepare_prefill, "rope": _prepare_rope, "step": _prepare_step,
}


# --------------------------------------------------------------------- run
def run(state):
    return _RUN[state["case"]["kind"]](state)


def _run_decode(s):
    out = s["attention"].decode_append(
        s["q"], s["key"][:, 0], s["value"][:, 0], s["tables"], s["context_lengths"], s["k"], s["v"], s["blocks"], s["offsets"],
        shared_prefix=s["groups"],
    )
    return {"out": out, "key": s["key"], "value": s["value"]}


def _run_prefill(s):
    return s["attention"].prefill(
        s["q"], s["key"][:, 0], s["value"][:, 0], s["tables"], s["context_lengths"], s["cu"], max(s["chunks"])
    )


def _run_rope(s):
    q = ops.rope_kv_append(
        s["key"], s["value"], 0, s["blocks"], s["offsets"], s["q"], s["k"], s["v"], s["cos"], s["sin"]
    )
    return {"q": q, "key": s["key"], "value": s["value"]}


def _run_step(s):
    rows = len(s["order"])
    ops.build_decode_metadata(
        s["descriptors"], rows, rows, s["tables"], PAGE, s["slots"], s["positions"], s["lengths"], s["blocks"], s["offsets"],
        s["row_tables"], s["width"],
    )
    outs = []
    for (key, value), q, k, v in zip(s["layers"], s["q"], s["k"], s["v"]):
        outs.append(s["attention"].decode_append(q, key, value, s["row_tables"], s["lengths"], k, v, s["blocks"], s["offsets"]))
    if len(s["exits"]):
        ops.kv_finalize(s["exits"], s["tables"], s["key"], s["value"], LOOPS)
    return {"outs": outs, "key": s["key"], "value": s["value"]}


_RUN = {"decode": _run_decode, "prefix": _run_decode, "prefill": _run_prefill, "rope": _run_rope, "step": _run_step}


# -------------------------------------------------------------------- work
def work(case):
    e = _esize(case)
    qrow = case["hq"] * case["d"] * e
    kvrow = 2 * case["hkv"] * case["d"] * e  # K and V of one token
    per_key = 4 * case["hq"] * case["d"]  # flops of one query row against one key
    if case["kind"] == "rope":
        rows = case["rows"]
        return dict(bytes=rows * (2 * qrow + 2 * kvrow + 2 * case["d"] * e + 16), flops=6 * rows * (case["hq"] + case["hkv"]) * case["d"])
    if case["kind"] == "prefill":
        pairs = _chunks(case)
        keys = sum(p + c for p, c in pairs)
        rows = sum(c for _, c in pairs)
        visible = sum(p * c + c * (c + 1) // 2 for p, c in pairs)
        return dict(bytes=keys * kvrow + 2 * rows * qrow + 4 * sum(_pages(p + c) for p, c in pairs), flops=per_key * visible)
    contexts = _contexts(case)
    rows, keys = len(contexts), sum(contexts)
    read = keys
    if case["kind"] == "prefix":  # a plane's prefix is read once, however many rows share it
        used = len({d % case["planes"] for d in _depths(case)})
        shared = case["prefix"] // PAGE * PAGE
        read = keys - rows * shared + used * shared
    one = dict(
        bytes=read * kvrow + rows * (2 * kvrow + 2 * qrow) + 4 * sum(_pages(n + 1) for n in contexts) + 20 * rows,
        flops=per_key * (keys + rows),
    )
    if case["kind"] == "decode" or case["kind"] == "prefix":
        return one
    copies = sum(LOOPS - 1 - d for _, d in _exits(case))
    return dict(bytes=LAYERS * (one["bytes"] + 2 * copies * kvrow), flops=LAYERS * one["flops"])


def tolerance(case):
    """Measured against 64 bits: about four times the present error of each storage type."""
    if case["kind"] == "rope":
        return "exact"  # one rounding per product and sum, as the elementwise operations round
    return {"bf16": {"rel": 1e-2}, "fp16": {"rel": 1.5e-3}, "fp32": {"rel": 1e-6}}[case["dtype"]]


# ------------------------------------------------------------------- exact
def _attention(q, k, v, visible):
    """q [n, hq, d] against k, v [keys, hkv, d]; query i sees the first visible[i] keys.  64 bits."""
    n, hq, d = q.shape
    group = hq // k.shape[1]
    qh = q.double().transpose(0, 1)  # [hq, n, d]
    kh = k.double().transpose(0, 1).repeat_interleave(group, dim=0)
    vh = v.double().transpose(0, 1).repeat_interleave(group, dim=0)
    mask = torch.arange(k.shape[0], device=q.device)[None, :] >= visible[:, None]
    out = torch.empty(n, hq, d, dtype=torch.float64, device=q.device)
    for h in range(hq):
        scores = (qh[h] @ kh[h].T.contiguous()) / math.sqrt(d)
        out[:, h] = torch.softmax(scores.masked_fill(mask, -math.inf), dim=-1) @ vh[h]
    return out


def _history(pool, table, n):
    return pool[table[: _pages(n)].long()].flatten(0, 1)[:n]


def _exact_rows(q, key, value, tables, lengths):
    rows = []
    for r, n in enumerate(lengths):
        k, v = _history(key, tables[r], n), _history(value, tables[r], n)
        rows.append(_attention(q[r : r + 1], k, v, torch.tensor([n], device=q.device)))
    return torch.cat(rows)


def exact(case, seed):
    s = prepare(case, seed)
    key, value = s["key"], s["value"]
    if case["kind"] == "prefill":
        outs, at = [], 0
        for i, (n, c) in enumerate(zip(s["lengths"], s["chunks"])):
            k, v = _history(key[:, 0], s["tables"][i], n), _history(value[:, 0], s["tables"][i], n)
            visible = torch.arange(n - c + 1, n + 1, device=k.device)
            outs.append(_attention(s["q"][at : at + c], k, v, visible))
            at += c
        return torch.cat(outs)
    if case["kind"] == "rope":
        cos, sin = s["cos"].double()[:, None], s["sin"].double()[:, None]

        def rotate(x):
            x = x.double()
            lo, hi = x.chunk(2, dim=-1)
            return x * cos + torch.cat([-hi, lo], dim=-1) * sin

        key = key.double()
        key[s["blocks"], 0, s["offsets"]] = rotate(s["k"])
        value[s["blocks"], 0, s["offsets"]] = s["v"]
        return {"q": rotate(s["q"]), "key": key, "value": value}
    if case["kind"] != "step":
        key[s["blocks"], 0, s["offsets"]] = s["k"]
        value[s["blocks"], 0, s["offsets"]] = s["v"]
        return {"out": _exact_rows(s["q"], key[:, 0], value[:, 0], s["tables"], s["lengths"]), "key": key, "value": value}
    contexts, depths = _contexts(case), _depths(case)
    lengths = [contexts[i] + 1 for i in s["order"]]
    tables = torch.stack([s["tables"][i, depths[i]] for i in s["order"]])
    outs = []
    for layer in range(LAYERS):
        for r, n in enumerate(lengths):
            block, offset = int(tables[r, (n - 1) // PAGE]), (n - 1) % PAGE
            key[block, layer, offset] = s["k"][layer][r]
            value[block, layer, offset] = s["v"][layer][r]
        outs.append(_exact_rows(s["q"][layer], key[:, layer], value[:, layer], tables, lengths))
    for slot, depth in _exits(case):
        page, offset = divmod(contexts[slot], PAGE)
        table = s["tables"][slot, :, page].tolist()
        for target in range(depth + 1, LOOPS):
            key[table[target], :, offset] = key[table[depth], :, offset]
            value[table[target], :, offset] = value[table[depth], :, offset]
    return {"outs": outs, "key": key, "value": value}
