"""Performance cases: the work a user of this package has it do, through its
public entry points.

Six kinds of work, each over the range its sizes are drawn from:

``paged``    one layer's decode of a serving batch from device page pools
             (``decode_paged`` with a kept plan and page records), from one
             short sequence to long-context batches, in every page format;
             optionally with the append of the step's new token
``encode``   device encode of key and value rows into pages: a prefill's
             rows, or the rows of one decode step
``prefill``  ``DevicePagedKVCache``: ingest a prompt, then decode one query
``serve``    ``DeviceVllmPagedKVCache``: one continuous-batching step, the new
             token of every sequence written by slot mapping, then a decode
             by block tables
``grouped``  the backend's grouped decode over prepared pages, with or
             without logits and weights
``step``     ``decode_step``: one query over one KV head's prepared pages
``session``  ``PagedDecodeSession`` with a window and a page shortlist

Inputs are made on the GPU from the seed alone.  Page formats are written
"m3" (fp16 rows), "m3_i8", "m3_f32", or "<a|s><bits>g<group>" (M0 affine or
symmetric codes), for instance "a4g32".
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from dotcache_amd import attention_runtime, backends
from dotcache_amd.block_cache import DeviceVllmPagedKVCache
from dotcache_amd.config import DotCacheConfig
from dotcache_amd.decode import decode_paged, gather_records, plan_decode, workspace_bytes
from dotcache_amd.kv_cache import DevicePagedKVCache
from dotcache_amd.page_cache import PreparedPageCache
from dotcache_amd.page_pool import DevicePagePool, PoolGeometry, page_format_of
from dotcache_amd.session_runtime import PagedDecodeSession

_DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


# ---- page formats -----------------------------------------------------------
def _parse(fmt: str) -> dict:
    if fmt.startswith("m3"):
        return {"mode": "M3", "escape": {"m3": "float16", "m3_i8": "int8", "m3_f32": "float32"}[fmt], "group": 32}
    bits, group = fmt[1:].split("g")
    return {"mode": "M0", "scheme": "affine" if fmt[0] == "a" else "symmetric", "bits": int(bits), "group": int(group)}


def _pool_format(fmt: str) -> tuple[int, int]:
    f = _parse(fmt)
    return page_format_of(f["mode"], f.get("scheme", "affine"), f.get("bits", 4), f.get("escape", "float16"))


def _token_bytes(fmt: str, hd: int) -> float:
    """Compressed bytes of one row."""
    f = _parse(fmt)
    if f["mode"] == "M3":
        return {"float16": 2 * hd, "float32": 4 * hd, "int8": hd + 2}[f["escape"]]
    groups = -(-hd // f["group"])
    words = -(-f["group"] * f["bits"] // 32)
    return groups * (4 * words + (4 if f["scheme"] == "affine" else 2))


def _quotient(a, b):
    """The correctly rounded fp32 quotient of two fp32 tensors, as fp64
    (a 53-bit quotient rounded to 24 bits is the directly rounded one)."""
    return (a.double() / b.double()).float().double()


def _stored(x, fmt: str):
    """What a page of this format holds for fp32 rows ``x [..., hd]``, in
    fp64: codes by the page format's definition (fp32 scale, round half to
    even), then the fp16 scale and bias that are kept."""
    f = _parse(fmt)
    if f["mode"] == "M3":
        if f["escape"] == "float16":
            return x.half().double()
        if f["escape"] == "float32":
            return x.double()
        scale = _quotient(x.abs().amax(-1, keepdim=True), torch.tensor(127.0, device=x.device)).clamp_min(1e-8).half()
        return torch.round(_quotient(x, scale.float())).clamp(-127, 127) * scale.double()
    hd, gs, bits = x.shape[-1], f["group"], f["bits"]
    pad = -hd % gs
    g = torch.nn.functional.pad(x, (0, pad)).unflatten(-1, (-1, gs))
    if f["scheme"] == "affine":
        top = float((1 << bits) - 1)
        lo, hi = g.amin(-1, keepdim=True), g.amax(-1, keepdim=True)
        scale = _quotient(hi - lo, torch.tensor(top, device=x.device)).float().clamp_min(1e-8)
        code = torch.round(_quotient(g - lo, scale)).clamp(0, top)
        out = code * scale.half().double() + lo.half().double()
    else:
        qmax = float((1 << (bits - 1)) - 1)
        scale = _quotient(g.abs().amax(-1, keepdim=True), torch.tensor(max(qmax, 1.0), device=x.device))
        scale = scale.float().clamp_min(1e-8)
        out = torch.round(_quotient(g, scale)).clamp(-qmax, qmax) * scale.half().double()
    return out.flatten(-2)[..., :hd]


def _attend(q, k, v):
    """(logits, weights, output) in fp64 of queries [..., Q, hd] over rows [..., T, hd]."""
    logits = torch.matmul(q, k.transpose(-1, -2).contiguous())
    w = torch.softmax(logits, dim=-1)
    return logits, w, torch.matmul(w, v)


# ---- seeded inputs ------------------------------------------------------------
def _gen(seed: int, tag: int):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + tag)
    return g


def _rows(case: dict, seed: int, kind: str, b: int, heads: int, tokens: int):
    """fp32 rows [heads, tokens, hd] of sequence b: normal, optionally with
    four x16 outlier channels per head, or Student-t with 4 degrees of
    freedom per row; rounded to the case's row dtype."""
    gen = _gen(seed, 2 * b + (kind == "V"))
    hd = case["hd"]
    x = torch.randn((heads, tokens, hd), generator=gen, device="cuda")
    values = case.get("values", "normal")
    if values == "student_t":
        chi = torch.randn((4, heads, tokens, 1), generator=gen, device="cuda").square().sum(0)
        x = x / torch.sqrt(chi / 4.0)
    elif values == "outliers":
        gen = _gen(seed, -1 - (kind == "V"))
        channels = torch.rand((heads, hd), generator=gen, device="cuda").argsort(-1)[:, :4]
        scale = torch.ones((heads, hd), device="cuda").scatter_(1, channels, 16.0)
        x = x * scale[:, None, :]
    return x.to(_DTYPES[case.get("rows", "f32")]).float()


def _queries(case: dict, seed: int, *shape):
    q = torch.randn(shape, generator=_gen(seed, 1 << 20), device="cuda")
    return q.to(_DTYPES[case.get("queries", "f32")])


# ---- paged: one layer's decode over device pools ----------------------------
def _lengths(case: dict) -> list[int]:
    """Tokens of every sequence: equal, or log-uniform in the case's range
    (fixed by the case, so that its work is)."""
    if "ragged_low" not in case:
        return [case["context"]] * case["batch"]
    r = random.Random(case["batch"] * 7919 + case["context"])
    lo, hi = math.log(case["ragged_low"]), math.log(case["context"])
    return [int(math.exp(r.uniform(lo, hi))) for _ in range(case["batch"])]


def _page_format_at(case: dict, kind: str, h: int, page: int, pages: int) -> str:
    """Format of one page: exact (fp16) for the newest ``window_pages`` and,
    for keys, for the first ``exact_heads`` KV heads."""
    if page >= pages - case.get("window_pages", 0):
        return "m3"
    if kind == "K" and h < case.get("exact_heads", 0):
        return "m3"
    return case["key" if kind == "K" else "value"]


def _prepare_paged(case: dict, seed: int) -> dict:
    hd, H, P, lens = case["hd"], case["kv_heads"], case["page"], _lengths(case)
    B = len(lens)
    pages = [-(-n // P) for n in lens]
    pools, tables = {}, {}
    perm = random.Random(seed + 5)
    for kind in ("K", "V"):
        fmt = case["key" if kind == "K" else "value"]
        geo = PoolGeometry(hd, _parse(fmt)["group"], P, case.get("layout", "group_major"))
        at = [(b, h, p, _page_format_at(case, kind, h, p, pages[b]))
              for b in range(B) for h in range(H) for p in range(pages[b])]
        perm.shuffle(at)  # a pool whose pages came and went
        probe = DevicePagePool(geo, reserve_bytes=256, reserve_pages=16)
        sizes = {f: probe.blob_bytes(*_pool_format(f)) for f in sorted({a[3] for a in at})}
        pool = DevicePagePool(geo, reserve_bytes=sum(sizes[a[3]] for a in at) + 256, reserve_pages=len(at) + 16)
        table = np.zeros((B, H, max(pages)), dtype=np.int32)
        for f in sizes:
            mine = [a for a in at if a[3] == f]
            for (b, h, p, _), pid in zip(mine, pool.allocate(*_pool_format(f), len(mine), tokens=P).tolist()):
                table[b, h, p] = pid
        for b in range(B):
            pool.set_tokens(table[b, :, pages[b] - 1], lens[b] - (pages[b] - 1) * P)
        dev = torch.from_numpy(table).cuda()
        slot = torch.arange(max(lens), device="cuda", dtype=torch.int32)
        for b in range(B):
            n = lens[b]
            ids = dev[b][:, (slot[:n] // P).long()].reshape(-1)
            x = _rows(case, seed, kind, b, H, n)
            pool.encode_rows(x.reshape(H * n, hd), ids, (slot[:n] % P).repeat(H))
        pools[kind], tables[kind] = pool, (table, dev)
    n_q = case["q_per_kv"]
    last = np.asarray([n - (p - 1) * P for n, p in zip(lens, pages)], dtype=np.int32)
    seq_pages = np.asarray(pages, dtype=np.int32)
    (kt, k_dev), (vt, v_dev) = tables["K"], tables["V"]
    plan, _ = plan_decode(pools["K"], pools["V"], kt, vt, seq_pages, n_q, last_page_tokens=last)
    state = {
        "kind": "paged", "k_pool": pools["K"], "v_pool": pools["V"], "k_table": k_dev, "v_table": v_dev,
        "seq_pages": seq_pages, "plan": plan,
        "records": gather_records(pools["K"], k_dev, v_dev, seq_pages, plan, v_pool=pools["V"]),
        "queries": _queries(case, seed, B, H, n_q, hd), "scale": hd ** -0.5,
        "workspace": torch.empty(max(workspace_bytes(plan, n_q, hd), 16), dtype=torch.uint8, device="cuda"),
    }
    if case.get("append"):  # the newest token's row of every stream, encoded again into its slot each step
        new = {kind: torch.cat([_rows(case, seed, kind, b, H, n)[:, -1] for b, n in enumerate(lens)])
               for kind in ("K", "V")}
        tail = {kind: torch.from_numpy(np.stack([tables[kind][0][b, :, pages[b] - 1] for b in range(B)]).ravel()).cuda()
                for kind in ("K", "V")}
        slots = torch.from_numpy(np.repeat(last - 1, H).astype(np.int32)).cuda()
        state["append"] = (new["K"], new["V"], tail["K"], slots, tail["V"], slots)
    return state


def _run_paged(s: dict):
    if "append" in s:
        s["k_pool"].encode_rows_with(s["v_pool"], *s["append"])
    return decode_paged(s["k_pool"], s["k_table"], s["v_table"], s["seq_pages"], s["queries"], query_scale=s["scale"],
                        plan=s["plan"], workspace=s["workspace"], validate=False, v_pool=s["v_pool"],
                        records=s["records"])


def _exact_paged(case: dict, seed: int):
    hd, H, P, n_q, lens = case["hd"], case["kv_heads"], case["page"], case["q_per_kv"], _lengths(case)
    q = _queries(case, seed, len(lens), H, n_q, hd).double() * hd ** -0.5
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for b, n in enumerate(lens):
        pages = -(-n // P)
        rows = {kind: _rows(case, seed, kind, b, H, n) for kind in ("K", "V")}
        for h in range(H):
            kv = []
            for kind in ("K", "V"):
                cut = min(n, max(pages - case.get("window_pages", 0), 0) * P)  # pages before the window
                parts = [_stored(rows[kind][h, a:e], _page_format_at(case, kind, h, a // P, pages))
                         for a, e in ((0, cut), (cut, n)) if e > a]
                kv.append(torch.cat(parts))
            out[b, h] = _attend(q[b, h], *kv)[2]
    return out


# ---- encode: rows into pages -------------------------------------------------------
def _prepare_encode(case: dict, seed: int) -> dict:
    hd, H, P, T, B = case["hd"], case["kv_heads"], case["page"], case["tokens"], case["batch"]
    rows, pools, dest = [], [], []
    for kind in ("K", "V"):
        fmt = case["key" if kind == "K" else "value"]
        geo = PoolGeometry(hd, _parse(fmt)["group"], P)
        pages = B * H * -(-T // P)
        probe = DevicePagePool(geo, reserve_bytes=256, reserve_pages=16)
        pool = DevicePagePool(geo, reserve_bytes=pages * probe.blob_bytes(*_pool_format(fmt)), reserve_pages=pages)
        ids = pool.allocate(*_pool_format(fmt), pages, tokens=min(T, P)).reshape(B * H, -1)
        token = torch.arange(T, device="cuda", dtype=torch.int32)
        x = torch.stack([_rows(case, seed, kind, b, H, T) for b in range(B)]).reshape(-1, hd)
        rows.append(x.to(_DTYPES[case["rows"]]).contiguous())
        pools.append(pool)
        dest += [torch.from_numpy(ids).cuda()[:, (token // P).long()].reshape(-1).contiguous(), (token % P).repeat(B * H)]
    return {"kind": "encode", "rows": rows, "pools": pools, "dest": dest}


def _run_encode(s: dict):
    s["pools"][0].encode_rows_with(s["pools"][1], *s["rows"], *s["dest"])
    return [pool.arena for pool in s["pools"]]


# ---- caches: a prompt's ingest, a serving step -------------------------------------
def _config(case: dict) -> DotCacheConfig:
    k, v = _parse(case["key"]), _parse(case["value"])
    return DotCacheConfig(head_dim=case["hd"], group_size=v["group"], tokens_per_page=case["page"],
                          bits_k=k.get("bits", 4), bits_v=v.get("bits", 4), default_mode_k=k["mode"],
                          default_mode_v=v["mode"], quant_scheme_k=k.get("scheme", "affine"),
                          quant_scheme_v=v.get("scheme", "affine"))


def _cached(case: dict, kind: str, x):
    """Rows [H, T, hd] as the caches hold them: full pages in the layer's
    format, the tail exact."""
    full = x.shape[1] // case["page"] * case["page"]
    return torch.cat([_stored(x[:, :full], case["key" if kind == "K" else "value"]), _stored(x[:, full:], "m3")], dim=1)


def _exact_cached(case: dict, seed: int, batch: int, tokens: int):
    H, n_q, hd = case["kv_heads"], case["q_per_kv"], case["hd"]
    q = _queries(case, seed, batch, H * n_q, hd).double().reshape(batch, H, n_q, hd) * hd ** -0.5
    return torch.stack([_attend(q[b], *(_cached(case, kind, _rows(case, seed, kind, b, H, tokens)) for kind in ("K", "V")))[2]
                        for b in range(batch)]).reshape(batch, H * n_q, hd)


def _prepare_prefill(case: dict, seed: int) -> dict:
    B, H, T = case["batch"], case["kv_heads"], case["tokens"]
    cache = DevicePagedKVCache(_config(case), num_hidden_layers=1, num_attention_heads=H * case["q_per_kv"],
                               num_key_value_heads=H, batch_size=B, reserve_pages_per_stream=T // case["page"] + 2)
    prompt = [torch.stack([_rows(case, seed, kind, b, H, T) for b in range(B)]).to(_DTYPES[case["rows"]])
              for kind in ("K", "V")]
    return {"kind": "prefill", "cache": cache, "prompt": prompt, "scale": case["hd"] ** -0.5,
            "queries": _queries(case, seed, B, H * case["q_per_kv"], case["hd"])}


def _run_prefill(s: dict):
    s["cache"].ingest_prefill_cache(0, *s["prompt"])
    return s["cache"].decode_layer(0, s["queries"], query_scale=s["scale"])


def _prepare_serve(case: dict, seed: int) -> dict:
    B, H, P, blocks = case["batch"], case["kv_heads"], case["page"], case["blocks"]
    cache = DeviceVllmPagedKVCache(config=_config(case), num_hidden_layers=1, num_attention_heads=H * case["q_per_kv"],
                                   num_key_value_heads=H, block_size=P, reserve_blocks=B * (blocks + 1))
    order = list(range(B * (blocks + 1)))
    random.Random(seed).shuffle(order)
    table = np.asarray(order, dtype=np.int64).reshape(B, blocks + 1)
    new = []
    for b in range(B):
        x = {kind: _rows(case, seed, kind, b, H, blocks * P + 1).transpose(0, 1).contiguous() for kind in ("K", "V")}
        slots = (table[b, :-1, None] * P + np.arange(P)).ravel()
        cache.write_slots(0, x["K"][:-1], x["V"][:-1], slots)
        new.append((x["K"][-1], x["V"][-1]))
    dt = _DTYPES[case["rows"]]
    return {"kind": "serve", "cache": cache, "keys": torch.stack([k for k, _ in new]).to(dt),
            "values": torch.stack([v for _, v in new]).to(dt), "slots": table[:, -1] * P, "table": torch.from_numpy(table),
            "lens": torch.full((B,), blocks * P + 1), "scale": case["hd"] ** -0.5,
            "queries": _queries(case, seed, B, H * case["q_per_kv"], case["hd"])}


def _run_serve(s: dict):
    # every sequence's new token opens its next block, so the step can be repeated
    s["cache"].write_slots(0, s["keys"], s["values"], s["slots"])
    return s["cache"].decode_block_tables(0, s["queries"], s["table"], s["lens"], query_scale=s["scale"])


# ---- prepared pages: the backend functions and the session ---------------------------
def _host_pages(case: dict, kind: str, x):
    """Rows [T, hd] as host pages, encoded on the device."""
    fmt = case["key" if kind == "K" else "value"]
    P, T, hd = case["page"], x.shape[0], case["hd"]
    n = -(-T // P)
    pool = DevicePagePool(PoolGeometry(hd, _parse(fmt)["group"], P), reserve_bytes=n * P * hd * 4 + 256, reserve_pages=n)
    ids = pool.allocate(*_pool_format(fmt), n, tokens=P)
    pool.set_tokens(ids[-1:], T - (n - 1) * P)
    token = torch.arange(T, device="cuda", dtype=torch.int32)
    pool.encode_rows(x, torch.from_numpy(ids).cuda()[(token // P).long()], token % P)
    pages = [pool.download_page(int(i), kind=kind) for i in ids]
    for i, page in enumerate(pages):
        page.header.token_start = i * P
    return pages


def _page_groups(case: dict, seed: int, groups: int):
    out = []
    for kind in ("K", "V"):
        x = _rows(case, seed, kind, 0, groups, case["context"])
        out.append([_host_pages(case, kind, x[g]) for g in range(groups)])
    return out


def _prepare_grouped(case: dict, seed: int) -> dict:
    G = case["kv_heads"]
    keys, values = ([attention_runtime.prepare_pages(p, backend="hip_mi355x") for p in side]
                    for side in _page_groups(case, seed, G))
    q = _queries(case, seed, G, case["q_per_kv"], case["hd"]) * case["hd"] ** -0.5
    return {"kind": "grouped", "args": (list(q), keys, values), "logits": case["logits"]}


def _run_grouped(s: dict):
    if s["logits"]:
        return backends.decode_grouped_multiquery_step_prepared_hip_tensor(*s["args"])
    return backends.decode_grouped_multiquery_step_prepared_hip_tensor_output_only(*s["args"])


def _exact_grouped(case: dict, seed: int):
    G, hd = case["kv_heads"], case["hd"]
    q = (_queries(case, seed, G, case["q_per_kv"], hd) * hd ** -0.5).double()
    k, v = (_stored(_rows(case, seed, kind, 0, G, case["context"]), case[name])
            for kind, name in (("K", "key"), ("V", "value")))
    all_three = _attend(q, k, v)
    return all_three if case["logits"] else all_three[2]


def _prepare_step(case: dict, seed: int) -> dict:
    (keys,), (values,) = _page_groups(case, seed, 1)
    keys, values = (attention_runtime.prepare_pages(p, backend="hip_mi355x") for p in (keys, values))
    q = _queries(case, seed, case["hd"]) * case["hd"] ** -0.5
    return {"kind": "step", "args": (q.cpu().numpy(), keys, values)}


def _run_step(s: dict):
    return attention_runtime.decode_step(*s["args"], backend="hip_mi355x")


def _exact_step(case: dict, seed: int):
    q = (_queries(case, seed, case["hd"]) * case["hd"] ** -0.5).double()[None]
    k, v = (_stored(_rows(case, seed, kind, 0, 1, case["context"]), case[name])[0]
            for kind, name in (("K", "key"), ("V", "value")))
    return tuple(t[0] for t in _attend(q, k, v))


def _prepare_session(case: dict, seed: int) -> dict:
    (keys,), (values,) = _page_groups(case, seed, 1)
    session = PagedDecodeSession(backend="hip_mi355x", cache=PreparedPageCache(), recent_window_tokens=case["recent"],
                                 sink_window_tokens=case["sink"], relevance_top_k=case["top_k"],
                                 relevance_sketch_size=case["sketch"], relevance_mode=case["mode"])
    session.preload(keys, values)
    q = _queries(case, seed, case["hd"]) * case["hd"] ** -0.5
    return {"kind": "session", "session": session, "query": q.cpu().numpy()}


def _run_session(s: dict):
    return s["session"].decode(s["query"])


def _exact_session(case: dict, seed: int):
    P, n = case["page"], case["context"] // case["page"]
    q = (_queries(case, seed, case["hd"]) * case["hd"] ** -0.5).double()
    k, v = (_stored(_rows(case, seed, kind, 0, 1, n * P), case[name])[0].reshape(n, P, -1)
            for kind, name in (("K", "key"), ("V", "value")))
    if case["mode"] == "sketch":
        sketch = torch.stack([c.mean(1) for c in torch.tensor_split(k, case["sketch"], dim=1)], dim=1)
        score = (sketch @ q).amax(1)
    else:
        score = k.amax(1) @ q.clamp_min(0) + k.amin(1) @ q.clamp_max(0)
    start = torch.arange(n, device="cuda") * P
    window = (start < case["sink"]) | (start + P > n * P - case["recent"])
    best = torch.argsort(score.masked_fill(window, -math.inf), descending=True, stable=True)[: case["top_k"]]
    window[best] = True
    return tuple(t[0] for t in _attend(q[None], k[window].flatten(0, 1), v[window].flatten(0, 1)))


# ---- the cases -----------------------------------------------------------------------
def listed() -> list[dict]:
    return [
        # The smallest serving call: one sequence of 4096 tokens on a 1B-shaped
        # layer (8 KV heads x 4 queries, head_dim 64, 4-bit affine pages).
        {"name": "decode_b1_4k", "kind": "paged", "batch": 1, "context": 4096, "kv_heads": 8, "q_per_kv": 4, "hd": 64,
         "page": 64, "key": "a4g32", "value": "a4g32", "queries": "bf16"},
        # The headline: a 7B-shaped GQA layer, 8 x 16384 tokens, exact keys and
        # 4-bit symmetric values, keys and values with outlier channels.
        {"name": "decode_b8_16k", "kind": "paged", "batch": 8, "context": 16384, "kv_heads": 4, "q_per_kv": 7, "hd": 128,
         "page": 64, "key": "m3", "value": "s4g32", "queries": "bf16", "values": "outliers"},
        # Continuous batching: 64 sequences of 256 to 32768 tokens, odd lengths,
        # one of the two KV heads' keys kept exact by the sensitivity map.
        {"name": "decode_ragged_b64", "kind": "paged", "batch": 64, "context": 32768, "ragged_low": 256, "kv_heads": 2,
         "q_per_kv": 6, "hd": 128, "page": 64, "key": "a4g32", "value": "s8g64", "exact_heads": 1, "queries": "bf16"},
        # Long context: 4 x 131072 tokens at head_dim 256, 4-bit pages with an
        # exact recent page, and the append of the step's token.
        {"name": "append_decode_b4_128k", "kind": "paged", "batch": 4, "context": 131072 + 64, "kv_heads": 4,
         "q_per_kv": 4, "hd": 256, "page": 128, "key": "a4g32", "value": "a4g32", "window_pages": 1, "append": True,
         "queries": "bf16", "values": "student_t"},
        # The compact tiers: int8 escape keys, 3-bit values.
        {"name": "decode_int8_3bit_b4_8k", "kind": "paged", "batch": 4, "context": 8192, "kv_heads": 4, "q_per_kv": 4,
         "hd": 128, "page": 64, "key": "m3_i8", "value": "a3g32", "queries": "bf16"},
        # A head_dim that is no power of two, an odd context, a small batch.
        {"name": "decode_hd96_b3_3k", "kind": "paged", "batch": 3, "context": 2901, "kv_heads": 6, "q_per_kv": 2, "hd": 96,
         "page": 64, "key": "a4g32", "value": "a4g32", "queries": "f16"},
        # The prefill's encode of one 7B-shaped layer: 8 x 16384 bf16 rows of
        # 4 KV heads into exact keys and 4-bit values.
        {"name": "encode_b8_16k", "kind": "encode", "batch": 8, "tokens": 16384, "kv_heads": 4, "hd": 128, "page": 64,
         "key": "m3", "value": "s4g32", "rows": "bf16", "values": "outliers"},
        # A prompt into the model cache, with a tail, and its first decode.
        {"name": "prefill_b2_4k", "kind": "prefill", "batch": 2, "tokens": 4109, "kv_heads": 4, "q_per_kv": 7, "hd": 128,
         "page": 64, "key": "a4g32", "value": "a4g32", "rows": "bf16", "queries": "bf16"},
        # One step of a serving engine: 16 sequences' new tokens, then their decode.
        {"name": "serve_b16_2k", "kind": "serve", "batch": 16, "blocks": 32, "kv_heads": 8, "q_per_kv": 4, "hd": 64,
         "page": 64, "key": "a4g32", "value": "a4g32", "rows": "bf16", "queries": "bf16"},
        # The backend's grouped decode with logits and weights: a 3B-shaped
        # layer (8 KV heads x 3 queries) over 4096 tokens.
        {"name": "grouped_logits_4k", "kind": "grouped", "context": 4096, "kv_heads": 8, "q_per_kv": 3, "hd": 128,
         "page": 64, "key": "a4g32", "value": "a4g32", "logits": True},
        # One query over one head's 4096 tokens, results on the host: the
        # reference's own latency ladder.
        {"name": "step_4k", "kind": "step", "context": 4096, "hd": 128, "page": 64, "key": "a4g32", "value": "a4g32"},
        # A session over 32768 tokens that attends a window and 64 shortlisted pages.
        {"name": "session_32k_top64", "kind": "session", "context": 32768, "hd": 128, "page": 64, "key": "a4g32",
         "value": "a4g32", "sink": 64, "recent": 1024, "top_k": 64, "sketch": 4, "mode": "sketch"},
    ]


_KEYS = ["a4g32", "m3", "s4g32", "a8g32", "a3g32", "a2g32", "m3_i8", "a4g16", "m3_f32"]
_VALUES = ["a4g32", "s4g32", "s8g64", "a8g32", "a3g32", "s2g32", "m3", "m3_i8", "a4g16"]


def draw(rng: random.Random) -> dict:
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["paged", "paged", "paged", "encode", "prefill", "serve", "grouped", "step", "session"])
    hd = rng.choice([64, 96, 128, 128, 256])
    case = {"kind": kind, "hd": hd, "page": rng.choice([32, 64, 64, 128])}
    if kind == "paged":
        case.update(kv_heads=rng.choice([1, 2, 4, 8]), q_per_kv=rng.choice([1, 2, 3, 4, 6, 7, 8, 16]),
                    queries=rng.choice(["bf16", "f16", "f32"]), values=rng.choice(["normal", "outliers", "student_t"]),
                    key=rng.choice(_KEYS), value=rng.choice(_VALUES))
        case["batch"] = size(1, 64)
        # from 100 tokens up; in all an eighth of the largest listed case's values (its formats are the smallest)
        case["context"] = size(100, min(131072, (1 << 26) // (case["batch"] * case["kv_heads"] * hd)))
        if rng.random() < 0.4 and case["batch"] > 1:
            case["ragged_low"] = max(1, case["context"] // rng.choice([2, 16, 128]))
        if rng.random() < 0.3:
            case["exact_heads"] = rng.randint(0, case["kv_heads"])
        if rng.random() < 0.3:
            case.update(window_pages=1, append=True)
    elif kind == "encode":
        case.update(kv_heads=rng.choice([1, 2, 4, 8]), batch=size(1, 64), key=rng.choice(_KEYS), value=rng.choice(_VALUES),
                    rows=rng.choice(["bf16", "f16", "f32"]), values=rng.choice(["normal", "outliers"]))
        case["tokens"] = 1 if rng.random() < 0.3 else size(2, min(32768, (1 << 26) // (case["batch"] * case["kv_heads"] * hd)))
    elif kind == "prefill":
        case.update(kv_heads=rng.choice([2, 4, 8]), q_per_kv=rng.choice([1, 4, 7]), batch=rng.choice([1, 2]),
                    key=rng.choice(["a4g32", "m3", "a3g32"]), value=rng.choice(["a4g32", "s4g32"]),
                    rows=rng.choice(["bf16", "f32"]), queries="bf16", tokens=size(100, 4000))
    elif kind == "serve":
        case.update(kv_heads=rng.choice([2, 4, 8]), q_per_kv=rng.choice([1, 4, 7]), batch=size(1, 16),
                    key=rng.choice(["a4g32", "m3"]), value=rng.choice(["a4g32", "s4g32"]),
                    rows="bf16", queries="bf16", blocks=size(1, 32))
    else:
        case.update(context=size(100, 4096), key=rng.choice(["a4g32", "m3", "s8g32", "a3g32"]),
                    value=rng.choice(["a4g32", "s8g64", "m3"]))
        if kind == "grouped":
            case.update(kv_heads=rng.choice([1, 2, 8]), q_per_kv=rng.choice([1, 3, 4, 7]), logits=rng.random() < 0.5)
        elif kind == "session":
            case["context"] = case["page"] * size(8, 16384 // case["page"])
            case.update(sink=case["page"], recent=case["page"] * rng.randint(1, 4), top_k=rng.choice([1, 4, 16, 64]),
                        sketch=rng.choice([1, 2, 4]), mode=rng.choice(["sketch", "envelope"]))
    return case


_PREPARE = {"paged": _prepare_paged, "encode": _prepare_encode, "prefill": _prepare_prefill, "serve": _prepare_serve,
            "grouped": _prepare_grouped, "step": _prepare_step, "session": _prepare_session}
_RUN = {"paged": _run_paged, "encode": _run_encode, "prefill": _run_prefill, "serve": _run_serve,
        "grouped": _run_grouped, "step": _run_step, "session": _run_session}


def prepare(case: dict, seed: int) -> dict:
    return _PREPARE[case["kind"]](case, seed)


def run(state: dict):
    return _RUN[state["kind"]](state)


def work(case: dict) -> dict:
    kind, hd = case["kind"], case["hd"]
    k, v = (_token_bytes(case[name], hd) for name in ("key", "value"))
    if kind == "encode":
        rows = case["batch"] * case["kv_heads"] * case["tokens"]
        in_bytes = 4 if case["rows"] == "f32" else 2
        return {"bytes": int(rows * (2 * hd * in_bytes + 16 + k + v)), "flops": 8 * rows * hd}
    if kind == "paged":
        lens, H, n_q = _lengths(case), case["kv_heads"], case["q_per_kv"]
        nbytes = flops = 0
        for n in lens:
            window = min(n, case.get("window_pages", 0) * case["page"])
            exact = case.get("exact_heads", 0)
            nbytes += window * H * 4 * hd + (n - window) * (exact * 2 * hd + (H - exact) * k + H * v)
            flops += 4 * n * H * n_q * hd
        q_bytes = 4 if case["queries"] == "f32" else 2
        return {"bytes": int(nbytes + len(lens) * H * n_q * hd * (4 + q_bytes)), "flops": flops}
    H, n_q = case.get("kv_heads", 1), case.get("q_per_kv", 1)
    if kind == "prefill":
        rows, streams = case["batch"] * H * case["tokens"], case["batch"] * H
        in_bytes = 4 if case["rows"] == "f32" else 2
        # the prompt read, its pages written and read back by the decode
        return {"bytes": int(rows * (2 * hd * in_bytes + 2 * (k + v)) + streams * n_q * hd * 6),
                "flops": 8 * rows * hd + 4 * rows * n_q * hd}
    if kind == "serve":
        streams = case["batch"] * H
        rows = streams * (case["blocks"] * case["page"] + 1)
        return {"bytes": int(rows * (k + v) + streams * hd * (8 + 6 * n_q)), "flops": 4 * rows * n_q * hd}
    tokens = case["context"]
    summaries = 0
    if kind == "session":
        pages = case["context"] // case["page"]
        summaries = pages * 4 * hd * (case["sketch"] if case["mode"] == "sketch" else 2)
        tokens = min(pages, case["top_k"] + (case["sink"] + case["recent"]) // case["page"]) * case["page"]
    results = 8 * tokens * n_q if kind != "grouped" or case["logits"] else 0
    return {"bytes": int(H * (tokens * (k + v) + results + 8 * n_q * hd) + summaries),
            "flops": 4 * tokens * H * n_q * hd + summaries // 2}


def tolerance(case: dict):
    if case["kind"] == "encode":
        return "exact"  # the page format fixes every code, scale and bias
    # fp32 sums in another order and two-part fp16 operands: up to 2.8e-6 and 2e-5 from fp64 over these ranges
    return {"rel": 1e-5, "max": 1e-4}


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "encode":
        return None
    if kind == "paged":
        return _exact_paged(case, seed)
    if kind == "prefill":
        return _exact_cached(case, seed, case["batch"], case["tokens"])
    if kind == "serve":
        return _exact_cached(case, seed, case["batch"], case["blocks"] * case["page"] + 1)
    return {"grouped": _exact_grouped, "step": _exact_step, "session": _exact_session}[kind](case, seed)
