"""Block-table KV cache for a paged serving engine: vLLM block ids mapped
to device pages.

MI355X counterpart of the reference's vLLM adapter cache (reference
``dotcache/integrations/vllm_adapter/block_cache.py:92-551``).  The
reference keeps a ``ModelPagedKVCache`` per model and, beside it, one host
``EncodedPage`` per (layer, KV head, block id), re-encoded with numpy on
every appended token.  Here a block id owns device pages directly:

* a live (partially filled) block is an escape (M3) page per KV head,
  written row by row by ``dc_encode_rows``, plus its rows in fp32 in HBM;
* when its last slot is written the block is encoded, on the device, into
  a page of the layer's mode (``DotCacheConfig.resolve_page_mode``) from
  the fp32 rows -- bit-identical to the reference's ``encode_page`` of the
  block -- and the escape pages are released.

``write_slots`` takes rows with a vLLM-style slot mapping (``block_id *
block_size + offset``), and ``decode_block_tables`` decodes a batch of
sequences given by block tables and context lengths in one launch.  The
reference's single-sequence interface (``sync_layer_blocks``,
``append_step``, ``append_tokens_torch``, ``decode_layer``,
``block_entry``) is built on these two.
"""
from __future__ import annotations

from dataclasses import dataclass

import numpy as np

from .config import DotCacheConfig
from .decode import decode_paged, plan_decode, workspace_bytes
from .encode import resolve_encode_spec
from .kv_cache import default_q_head_to_kv_head
from .page_pool import DevicePagePool, PoolGeometry, page_format_of
from .types import EncodedPage


def _torch():
    import torch

    return torch


@dataclass(frozen=True)
class VllmBlockKey:
    """Reference ``block_cache.py:16-21``."""
    layer_id: int
    kv_head_id: int
    block_id: int
    kind: str


@dataclass
class VllmBlockEntry:
    """Reference ``block_cache.py:24-30``; ``page`` is read back from the
    device when the entry is requested."""
    key: VllmBlockKey
    page: EncodedPage
    finalized: bool
    token_count: int
    token_start: int


class DeviceVllmPagedKVCache:
    """Pages of ``num_hidden_layers`` layers addressed by block id.

    Rows may be numpy arrays or torch tensors (fp32, fp16, bf16), read as
    fp32.  ``block_size`` equals ``config.tokens_per_page``, as in the
    reference (``block_cache.py:103-104``).
    """

    def __init__(self, *, config: DotCacheConfig, num_hidden_layers: int, num_attention_heads: int,
                 num_key_value_heads: int, block_size: int, device="cuda", reserve_blocks: int = 64):
        torch = _torch()
        if config.tokens_per_page != block_size:
            raise ValueError("DotCache tokens_per_page must equal the vLLM block_size for this phase")
        q_map = default_q_head_to_kv_head(num_attention_heads, num_key_value_heads)
        if num_attention_heads // num_key_value_heads > 16:
            raise ValueError("at most 16 query heads per KV head")
        self.config = config
        self.block_size = int(block_size)
        self.num_hidden_layers = int(num_hidden_layers)
        self.num_attention_heads = int(num_attention_heads)
        self.num_key_value_heads = int(num_key_value_heads)
        self.device = torch.device(device)
        self.default_q_head_to_kv_head = q_map
        L, H, P, hd = self.num_hidden_layers, self.num_key_value_heads, self.block_size, config.head_dim
        self._specs = {kind: resolve_encode_spec(config, kind=kind) for kind in ("K", "V")}
        self._live_fmt = {kind: page_format_of("M3", "affine", 4, self._specs[kind]["escape_dtype"]) for kind in ("K", "V")}
        self._pools = {}
        for kind in ("K", "V"):
            geo = PoolGeometry(hd, config.group_size, P, self._specs[kind]["layout"])
            probe = DevicePagePool(geo, device=self.device, reserve_bytes=256, reserve_pages=16)
            blob = max(probe.blob_bytes(*self._page_format(kind, 0, 0)), probe.blob_bytes(*self._live_fmt[kind]))
            self._pools[kind] = DevicePagePool(geo, device=self.device, reserve_bytes=L * H * reserve_blocks * blob + (1 << 20),
                                               reserve_pages=L * H * reserve_blocks + 16)
        self.k_pool, self.v_pool = self._pools["K"], self._pools["V"]
        n = max(int(reserve_blocks), 1)
        # per layer, per block id: page id of each KV head (-1: none), tokens written, finalised, first token
        self._map = {kind: [np.full((n, H), -1, dtype=np.int32) for _ in range(L)] for kind in ("K", "V")}
        self._fill = [np.zeros(n, dtype=np.int32) for _ in range(L)]
        self._final = [np.zeros(n, dtype=bool) for _ in range(L)]
        self._start = [np.full(n, -1, dtype=np.int64) for _ in range(L)]
        # fp32 rows of each layer's live blocks, [slots, 2, H, P, hd] on the device; live block id -> slot.
        # (One cache is used from one stream at a time, which a caller that moves to another stream orders:
        # the layers share the pools' blobs and the workspace.)
        self._row_store = [torch.empty((0, 2, H, P, hd), dtype=torch.float32, device=self.device) for _ in range(L)]
        self._row_slots = [dict() for _ in range(L)]
        self._free_slots: list[list[int]] = [[] for _ in range(L)]
        # the single-sequence view of the reference interface: block ids in token order, cached length
        self._seq_blocks = [[] for _ in range(L)]
        self._seq_len = np.zeros(L, dtype=np.int64)
        self._workspace = None

    # ---- formats and small helpers ------------------------------------------
    def _page_format(self, kind: str, layer_id: int, kv_head_id: int) -> tuple[int, int]:
        spec = self._specs[kind]
        mode = self.config.resolve_page_mode(kind=kind, layer_id=layer_id, kv_head_id=kv_head_id)
        return page_format_of(mode, spec["scheme"], spec["bits"], spec["escape_dtype"])

    def _check_layer(self, layer_id: int) -> int:
        lid = int(layer_id)
        if not 0 <= lid < self.num_hidden_layers:
            raise ValueError(f"layer_id {layer_id} out of range")
        return lid

    def _as_rows(self, x, name: str):
        """``x [n, H, hd]`` on the device in fp32, fp16 or bf16 (the encoder
        reads each exactly as fp32); other types become fp32."""
        torch = _torch()
        t = x if isinstance(x, torch.Tensor) else torch.from_numpy(np.ascontiguousarray(np.asarray(x, dtype=np.float32)))
        t = t.to(device=self.device)
        if t.dtype not in (torch.float32, torch.float16, torch.bfloat16):
            t = t.float()
        if t.dim() != 3 or t.shape[1] != self.num_key_value_heads or t.shape[2] != self.config.head_dim:
            raise ValueError(f"{name} must have shape [tokens, {self.num_key_value_heads}, {self.config.head_dim}]")
        return t

    def _grow(self, lid: int, block_id: int) -> None:
        n = self._fill[lid].shape[0]
        if block_id < n:
            return
        m = max(2 * n, block_id + 1)
        for kind in ("K", "V"):
            grown = np.full((m, self.num_key_value_heads), -1, dtype=np.int32)
            grown[:n] = self._map[kind][lid]
            self._map[kind][lid] = grown
        self._fill[lid] = np.concatenate([self._fill[lid], np.zeros(m - n, dtype=np.int32)])
        self._final[lid] = np.concatenate([self._final[lid], np.zeros(m - n, dtype=bool)])
        self._start[lid] = np.concatenate([self._start[lid], np.full(m - n, -1, dtype=np.int64)])

    def _release(self, lid: int, blocks) -> None:
        blocks = np.atleast_1d(np.asarray(blocks, dtype=np.int64))
        for kind in ("K", "V"):
            ids = self._map[kind][lid][blocks]
            self._pools[kind].free(ids[ids >= 0])
            self._map[kind][lid][blocks] = -1
        self._fill[lid][blocks] = 0
        self._final[lid][blocks] = False
        self._start[lid][blocks] = -1
        for blk in blocks.tolist():
            if blk in self._row_slots[lid]:
                self._free_slots[lid].append(self._row_slots[lid].pop(blk))

    def _take_slots(self, lid: int, blocks: list[int]) -> None:
        """An fp32 row slot for every block (the store doubles when none is free)."""
        free = self._free_slots[lid]
        short = len(blocks) - len(free)
        if short > 0:
            n = int(self._row_store[lid].shape[0])
            m = max(2 * n, n + short)
            self._replace_store(lid, m, n, slice(0, n))
            free.extend(range(m - 1, n - 1, -1))
        for blk in blocks:
            self._row_slots[lid][blk] = free.pop()

    def _replace_store(self, lid: int, slots: int, n: int, rows) -> None:
        """A row store of ``slots`` slots whose first n hold ``rows`` of the old one."""
        torch = _torch()
        store = self._row_store[lid]
        new = torch.empty((slots, *store.shape[1:]), dtype=torch.float32, device=self.device)
        if n:
            new[:n].copy_(store[rows])
        if store.device.type == "cuda":
            # (it may have been made on another stream, where its memory could be reused
            # before this stream has read it)
            store.record_stream(torch.cuda.current_stream(store.device))
        self._row_store[lid] = new

    def _shrink_store(self, lid: int) -> None:
        """Give row slots back: all of them once no block is live, all but twice
        the live blocks' when fewer than a quarter are in use."""
        slots = self._row_slots[lid]
        live = len(slots)
        if int(self._row_store[lid].shape[0]) <= 4 * live:
            return
        self._replace_store(lid, 2 * live, live, list(slots.values()))
        self._row_slots[lid] = {blk: i for i, blk in enumerate(slots)}
        self._free_slots[lid] = list(range(2 * live - 1, live - 1, -1))

    def _allocate_final(self, kind: str, lid: int, n: int) -> np.ndarray:
        """Page ids ``[n, H]`` in the layer's modes."""
        H, P = self.num_key_value_heads, self.block_size
        fmts = [self._page_format(kind, lid, h) for h in range(H)]
        ids = np.empty((n, H), dtype=np.int32)
        for f in set(fmts):
            heads = [h for h in range(H) if fmts[h] == f]
            ids[:, heads] = self._pools[kind].allocate(*f, n * len(heads), tokens=P).reshape(n, len(heads))
        return ids

    # ---- the serving interface -------------------------------------------------
    def write_slots(self, layer_id: int, key_rows, value_rows, slot_mapping, *, token_start: int | None = None) -> None:
        """Write ``[n, H, hd]`` rows to ``slot_mapping[i] = block * block_size
        + offset``.  Within a block, slots are written in order from its
        fill (a block whose offset 0 is written again starts over).  A block
        whose last slot is written is finalised.  ``token_start`` (optional)
        is the absolute position of row 0, kept for page headers."""
        torch = _torch()
        lid = self._check_layer(layer_id)
        keys = self._as_rows(key_rows, "key_rows")
        values = self._as_rows(value_rows, "value_rows")
        if keys.shape[0] != values.shape[0]:
            raise ValueError("key_rows and value_rows must hold the same number of tokens")
        slots = np.asarray(slot_mapping.detach().cpu().numpy() if isinstance(slot_mapping, torch.Tensor) else slot_mapping,
                           dtype=np.int64).reshape(-1)
        if slots.shape[0] != keys.shape[0]:
            raise ValueError("slot_mapping needs one slot per row")
        if np.any(slots < 0):
            raise ValueError("slots must be non-negative")
        P = self.block_size
        n = slots.shape[0]
        if n == 0:
            return
        if keys.dtype != values.dtype:
            keys, values = keys.float(), values.float()
        # runs of consecutive slots of one block
        blocks, offs = slots // P, slots % P
        ends = np.append(np.flatnonzero((np.diff(slots) != 1) | (np.diff(blocks) != 0)) + 1, n).tolist()
        runs: list[tuple[int, int, int, int]] = []  # (block, offset, first row, end row), checked
        fills: dict[int, int] = {}                  # fill of the blocks of `runs` once they are written
        restart: list[int] = []                     # blocks reused from their first slot
        i, error = 0, None
        for j in ends:
            blk, off = int(blocks[i]), int(offs[i])
            self._grow(lid, blk)
            if off == 0 and blk in fills:  # written and reused in one call: the rows so far land first
                self._write_runs(lid, runs, restart, keys, values, offs, token_start)
                runs, fills, restart = [], {}, []
            fill = fills.get(blk, int(self._fill[lid][blk]))
            if off == 0 and fill > 0:
                restart.append(blk)
                fill = 0
            if off != fill:
                error = ValueError(f"block {blk} holds {fill} tokens; slot offset {off} is out of order")
                break
            runs.append((blk, off, i, j))
            fills[blk] = off + j - i
            i = j
        self._write_runs(lid, runs, restart, keys, values, offs, token_start)
        if error is not None:
            raise error

    def _write_runs(self, lid: int, runs, restart, keys, values, offs: np.ndarray, token_start: int | None) -> None:
        """Rows of checked runs in one launch (two when blocks fill up).  A
        block written whole is encoded straight into its final pages; rows
        of a live block go to its escape pages and, in fp32, to its row
        slot; rows that fill a live block only to its row slot, from which
        the block is then encoded."""
        if restart:
            self._release(lid, restart)
        if not runs:
            self._shrink_store(lid)
            return
        P, H, hd = self.block_size, self.num_key_value_heads, self.config.head_dim
        blk = np.asarray([r[0] for r in runs], dtype=np.int64)
        off, first, end = (np.asarray([r[k] for r in runs], dtype=np.int64) for k in (1, 2, 3))
        full = off + end - first == P
        whole = full & (off == 0)
        fresh = (off == 0) & ~whole
        self._start[lid][blk[off == 0]] = -1 if token_start is None else int(token_start) + first[off == 0]
        for kind in ("K", "V"):
            pool, table = self._pools[kind], self._map[kind][lid]
            if whole.any():
                table[blk[whole]] = self._allocate_final(kind, lid, int(whole.sum()))
            if fresh.any():
                table[blk[fresh]] = pool.allocate(*self._live_fmt[kind], int(fresh.sum()) * H, tokens=0).reshape(-1, H)
            live = ~full
            if live.any():
                pool.set_tokens(table[blk[live]].ravel(), np.repeat((off + end - first)[live], H))
        self._take_slots(lid, blk[fresh].tolist())
        self._fill[lid][blk] = off + end - first
        self._final[lid][blk[whole]] = True

        # row (token i, head h): page ids (-1 where only the row slot takes it), slot, row of the store
        a, z = int(first[0]), int(end[-1])
        run = np.repeat(np.arange(len(runs)), end - first)
        slot = offs[a:z]
        heads = np.arange(H)
        ids = [np.where((full & ~whole)[run][:, None], -1, self._map[kind][lid][blk][run]) for kind in ("K", "V")]
        rows = self._row_slots[lid]
        stored = np.asarray([-1 if w else rows[b] for b, w in zip(blk.tolist(), whole.tolist())], dtype=np.int64)[run]
        keep = np.where(stored[:, None] < 0, -1, (stored[:, None] * 2 * H + heads) * P + slot[:, None])
        slots = np.repeat(slot, H)
        flat = self._row_store[lid].view(-1, hd)
        kept = None
        if not whole.all():
            kept = (flat[: flat.shape[0] - H * P], flat[H * P:], keep.ravel())
        self.k_pool.encode_rows_with(self.v_pool, keys[a:z].reshape(-1, hd), values[a:z].reshape(-1, hd), ids[0].ravel(),
                                     slots, ids[1].ravel(), slots, keep=kept)
        done = blk[full & ~whole]
        if done.size:
            self._finalise(lid, done)
        self._shrink_store(lid)

    def _finalise(self, lid: int, blocks: np.ndarray) -> None:
        """Encode full live blocks from their fp32 rows and release their
        escape pages and row slots."""
        torch = _torch()
        P, H, hd = self.block_size, self.num_key_value_heads, self.config.head_dim
        n = len(blocks)
        at = [self._row_slots[lid].pop(b) for b in blocks.tolist()]
        store = self._row_store[lid]
        rows = store[at[0]][:, None] if n == 1 else store[torch.as_tensor(at, device=self.device)].transpose(0, 1)
        new = {}
        for kind in ("K", "V"):
            old = self._map[kind][lid][blocks]
            new[kind] = self._allocate_final(kind, lid, n)
            self._pools[kind].free(old)
            self._map[kind][lid][blocks] = new[kind]
        tables = torch.from_numpy(np.stack([new["K"], new["V"]]).reshape(2, n * H, 1).astype(np.int32)).to(self.device)
        self.k_pool.encode_streams_with(self.v_pool, rows[0].reshape(n * H, P, hd), rows[1].reshape(n * H, P, hd), tables)
        self._free_slots[lid].extend(at)
        self._final[lid][blocks] = True

    def decode_block_tables(self, layer_id: int, queries, block_tables, context_lens, q_head_to_kv_head=None, *,
                            query_scale: float = 1.0):
        """Attention of ``queries [B, Hq, hd]`` over sequences given as
        ``block_tables [B, W]`` block ids and ``context_lens [B]``: one
        decode launch for the batch.  Block b of a sequence holds tokens
        ``[b * block_size, ...)``; its token count is the block's fill."""
        torch = _torch()
        lid = self._check_layer(layer_id)
        B, Hq, H, hd, P = None, self.num_attention_heads, self.num_key_value_heads, self.config.head_dim, self.block_size
        q = queries if isinstance(queries, torch.Tensor) else torch.from_numpy(np.ascontiguousarray(np.asarray(queries, dtype=np.float32)))
        q = q.to(self.device)
        if q.dtype not in (torch.float32, torch.float16, torch.bfloat16):
            q = q.float()
        B = int(q.shape[0])
        if q.dim() != 3 or tuple(q.shape[1:]) != (Hq, hd):
            raise ValueError(f"queries must have shape [batch, {Hq}, {hd}]")
        lens = np.asarray(context_lens.detach().cpu().numpy() if isinstance(context_lens, torch.Tensor) else context_lens,
                          dtype=np.int64).reshape(-1)
        if lens.shape != (B,) or np.any(lens <= 0):
            raise ValueError("context_lens needs one positive length per sequence")
        bt = block_tables if isinstance(block_tables, torch.Tensor) else torch.from_numpy(np.asarray(block_tables, dtype=np.int64))
        if bt.dim() != 2 or bt.shape[0] != B:
            raise ValueError("block_tables must have shape [batch, max_blocks]")
        n_blocks = -(-lens // P)
        if np.any(n_blocks > bt.shape[1]):
            raise ValueError("a context length needs more blocks than its block-table row holds")
        bt_host = bt.detach().cpu().numpy().astype(np.int64)
        nmap = self._fill[lid].shape[0]
        at = np.clip(bt_host, 0, nmap - 1)
        used = np.arange(bt_host.shape[1])[None, :] < n_blocks[:, None]
        unknown = (used & ((bt_host < 0) | (bt_host >= nmap) | (self._map["K"][lid][at, 0] < 0))).any(axis=1)
        held = np.where(used, self._fill[lid][at], 0).sum(axis=1)
        wrong = np.flatnonzero(unknown | (held != lens))
        if wrong.size:
            b = int(wrong[0])
            if unknown[b]:
                raise ValueError(f"sequence {b} names a block with no pages in layer {lid}")
            raise ValueError(f"sequence {b}: its blocks hold {int(held[b])} tokens, context_lens says {int(lens[b])}")
        # [B, H, W] page ids, keys and values
        kt, vt = (self._map[kind][lid][at].transpose(0, 2, 1) for kind in ("K", "V"))
        k_table, v_table = torch.from_numpy(np.ascontiguousarray(np.stack([kt, vt]))).to(self.device)
        qmap = self.default_q_head_to_kv_head if q_head_to_kv_head is None else np.asarray(q_head_to_kv_head, dtype=np.int64)
        if qmap.shape != (Hq,) or np.any(qmap < 0) or np.any(qmap >= H) or np.any(np.bincount(qmap, minlength=H) != Hq // H):
            raise ValueError("q_head_to_kv_head must give every KV head the same number of query heads")
        order = np.argsort(qmap, kind="stable")
        contiguous = np.array_equal(order, np.arange(Hq))
        order_t = None if contiguous else torch.from_numpy(order).to(self.device)
        qg = (q if contiguous else q[:, order_t]).reshape(B, H, Hq // H, hd)
        seq_pages = n_blocks.astype(np.int32)
        last_tokens = self._fill[lid][bt_host[np.arange(B), n_blocks - 1]]
        # (a sequence's live block is an fp16 page: the split-K merge attends
        # it, and the decode launch takes the instance of the full blocks)
        plan, masks = plan_decode(self.k_pool, self.v_pool, kt, vt, seq_pages, Hq // H, device=self.device,
                                  last_page_tokens=last_tokens)
        need = workspace_bytes(plan, Hq // H, hd)
        if self._workspace is None or self._workspace.numel() < need:
            self._workspace = torch.empty(max(need, 16), dtype=torch.uint8, device=self.device)
        out = decode_paged(self.k_pool, k_table, v_table, seq_pages, qg, query_scale=query_scale, plan=plan,
                           workspace=self._workspace, validate=False, v_pool=self.v_pool,
                           page_masks=masks).reshape(B, Hq, hd)
        if contiguous:
            return out
        res = torch.empty_like(out)
        res[:, order_t] = out
        return res

    # ---- the reference's single-sequence interface --------------------------
    def sync_layer_blocks(self, layer_id: int, key_blocks, value_blocks, *, block_ids=None,
                          live_block_token_count: int = 0) -> None:
        """Replace layer ``layer_id`` with ``[H, n_blocks, block_size, hd]``
        blocks (reference ``block_cache.py:152-301``): all full, or the last
        one live with ``live_block_token_count`` tokens."""
        torch = _torch()
        lid = self._check_layer(layer_id)
        P, H, hd = self.block_size, self.num_key_value_heads, self.config.head_dim
        kb = [key_blocks, value_blocks]
        for i, x in enumerate(kb):
            t = x if isinstance(x, torch.Tensor) else torch.from_numpy(np.ascontiguousarray(np.asarray(x, dtype=np.float32)))
            t = t.to(device=self.device, dtype=torch.float32)
            if t.dim() == 5:
                if t.shape[0] != 1:
                    raise ValueError("batch dimension must be 1")
                t = t[0]
            if t.dim() != 4 or t.shape[0] != H or t.shape[2] != P or t.shape[3] != hd:
                raise ValueError(f"{'key' if i == 0 else 'value'}_blocks must have shape [kv_heads, block_count, block_size, head_dim]")
            kb[i] = t
        keys, values = kb
        if keys.shape[1] != values.shape[1]:
            raise ValueError("key_blocks and value_blocks must contain the same number of blocks")
        n = int(keys.shape[1])
        ids = list(range(n)) if block_ids is None else [int(b) for b in block_ids]
        if len(ids) != n:
            raise ValueError("block_ids must align with the number of blocks")
        if len(set(ids)) != n:
            raise ValueError("block_ids must be unique")
        if not 0 <= int(live_block_token_count) <= P:
            raise ValueError("live_block_token_count must be in [0, block_size]")
        self.clear_layer(lid)
        live = int(live_block_token_count)
        finalised = n if live in (0, P) else n - 1
        for i, blk in enumerate(ids):
            cnt = P if i < finalised else live
            slots = blk * P + np.arange(cnt)
            self.write_slots(lid, keys[:, i, :cnt].transpose(0, 1), values[:, i, :cnt].transpose(0, 1), slots,
                             token_start=i * P)
        self._seq_blocks[lid] = ids
        self._seq_len[lid] = finalised * P + (live if finalised < n else 0)

    def append_step(self, layer_id: int, key_step, value_step, token_index: int) -> None:
        """Append ``[H, n, hd]`` rows at ``token_index`` (the cached length);
        token t goes to block ``t // block_size`` (reference
        ``block_cache.py:303-325``, ``:456-517``)."""
        torch = _torch()
        lid = self._check_layer(layer_id)
        rows = []
        for name, x in (("key_step", key_step), ("value_step", value_step)):
            t = x if isinstance(x, torch.Tensor) else torch.from_numpy(np.ascontiguousarray(np.asarray(x, dtype=np.float32)))
            t = t.to(device=self.device, dtype=torch.float32)
            if t.dim() == 4:
                if t.shape[0] != 1:
                    raise ValueError(f"{name} batch dimension must be 1")
                t = t[0]
            if t.dim() != 3 or t.shape[0] != self.num_key_value_heads or t.shape[2] != self.config.head_dim:
                raise ValueError(f"{name} must have shape [kv_heads, token_count, head_dim]")
            rows.append(t)
        if rows[0].shape[1] != rows[1].shape[1]:
            raise ValueError("key_step and value_step token counts must match")
        if int(token_index) != int(self._seq_len[lid]):
            raise ValueError(f"layer {lid} expected token_index {int(self._seq_len[lid])}, received {token_index}")
        n = int(rows[0].shape[1])
        pos = int(token_index) + np.arange(n)
        seq = self._seq_blocks[lid]
        live = seq[-1] if seq and self._fill[lid][seq[-1]] < self.block_size else None
        for blk in np.unique(pos // self.block_size).tolist():
            if blk == live:
                continue
            if blk in seq:
                raise ValueError(f"token {int(pos[0])} maps to block {blk}, which already holds earlier tokens of layer {lid}")
            seq.append(blk)
        self.write_slots(lid, rows[0].transpose(0, 1), rows[1].transpose(0, 1), pos, token_start=int(token_index))
        self._seq_len[lid] += n

    append_step_torch = append_step

    def append_tokens_torch(self, layer_id: int, key_rows, value_rows, token_positions) -> None:
        """``[n, H, hd]`` rows at contiguous positions, appended in chunks
        that end on block boundaries (reference ``block_cache.py:420-454``)."""
        torch = _torch()
        pos = token_positions.reshape(-1).detach().cpu().numpy().astype(np.int64) if isinstance(token_positions, torch.Tensor) \
            else np.asarray(token_positions, dtype=np.int64).reshape(-1)
        if pos.size == 0:
            return
        if not np.array_equal(pos, np.arange(int(pos[0]), int(pos[0]) + pos.size)):
            raise ValueError("token positions must be contiguous (one sequence)")
        k = self._as_rows(key_rows, "key_rows").transpose(0, 1)
        v = self._as_rows(value_rows, "value_rows").transpose(0, 1)
        off = 0
        while off < pos.size:
            t = int(pos[off])
            m = min(self.block_size - t % self.block_size, pos.size - off)
            self.append_step(layer_id, k[:, off:off + m], v[:, off:off + m], t)
            off += m

    def decode_layer_torch(self, layer_id: int, query_step, q_head_to_kv_head=None, *, query_scale: float = 1.0):
        """The layer's sequence (its blocks in token order) decoded for
        ``query_step [Hq, hd]``; fp32 ``[Hq, hd]`` on the device (reference
        ``block_cache.py:519-551``)."""
        torch = _torch()
        lid = self._check_layer(layer_id)
        if self._seq_len[lid] == 0:
            raise ValueError(f"layer {lid} has no cached tokens to decode against")
        q = query_step if isinstance(query_step, torch.Tensor) else torch.from_numpy(np.ascontiguousarray(np.asarray(query_step, dtype=np.float32)))
        table = np.asarray(self._seq_blocks[lid], dtype=np.int64)[None]
        return self.decode_block_tables(lid, q.reshape(1, *q.shape[-2:]), table, [int(self._seq_len[lid])],
                                        q_head_to_kv_head, query_scale=query_scale)[0]

    def decode_layer(self, layer_id: int, query_step, q_head_to_kv_head=None, *, query_scale: float = 1.0) -> np.ndarray:
        return self.decode_layer_torch(layer_id, query_step, q_head_to_kv_head, query_scale=query_scale).cpu().numpy()

    # ---- entries and bookkeeping ----------------------------------------------
    def block_entry(self, layer_id: int, kv_head_id: int, block_id: int, kind: str) -> VllmBlockEntry:
        """The page of one (layer, KV head, block), read back from the device."""
        lid, h, blk = self._check_layer(layer_id), int(kv_head_id), int(block_id)
        if kind not in ("K", "V"):
            raise ValueError("kind must be K or V")
        if blk >= self._fill[lid].shape[0] or self._map[kind][lid][blk, h] < 0:
            raise KeyError(VllmBlockKey(lid, h, blk, kind))
        pool = self._pools[kind]
        pid = int(self._map[kind][lid][blk, h])
        header = pool.header_of(pid, kind)
        start = int(self._start[lid][blk])
        header.layer_id, header.kv_head_id, header.token_start = lid, h, max(start, 0)
        page = pool.download_page(pid, header, kind=kind)
        return VllmBlockEntry(key=VllmBlockKey(lid, h, blk, kind), page=page, finalized=bool(self._final[lid][blk]),
                              token_count=int(self._fill[lid][blk]), token_start=max(start, 0))

    def block_entries_for_layer(self, layer_id: int, *, kind: str) -> list[VllmBlockEntry]:
        lid = self._check_layer(layer_id)
        blocks = np.flatnonzero(self._fill[lid] > 0).tolist()
        return [self.block_entry(lid, h, b, kind) for h in range(self.num_key_value_heads) for b in blocks]

    def clear_layer(self, layer_id: int) -> None:
        lid = self._check_layer(layer_id)
        self._release(lid, np.flatnonzero((self._map["K"][lid][:, 0] >= 0) | (self._fill[lid] > 0)))
        self._shrink_store(lid)
        self._seq_blocks[lid] = []
        self._seq_len[lid] = 0

    def clear(self) -> None:
        for lid in range(self.num_hidden_layers):
            self.clear_layer(lid)

    @property
    def resident_bytes(self) -> int:
        """Bytes of every block's pages (valid tokens only)."""
        total = 0
        for lid in range(self.num_hidden_layers):
            for kind in ("K", "V"):
                ids = self._map[kind][lid]
                total += self._pools[kind].read_bytes(ids[ids >= 0])
        return total


__all__ = ["DeviceVllmPagedKVCache", "VllmBlockEntry", "VllmBlockKey"]
