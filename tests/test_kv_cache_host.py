"""Host-side checks of the device KV cache that run before any device work:
argument validation and the token-index contract of ``append_step``
(reference ``model_kv_cache.py:3873-3876``)."""
import numpy as np
import pytest

from dotcache_amd.config import DotCacheConfig
from dotcache_amd.kv_cache import DevicePagedKVCache, default_q_head_to_kv_head


def _cache(**kw):
    cfg = DotCacheConfig(head_dim=64, group_size=32, tokens_per_page=16)
    args = dict(num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2, batch_size=1, device="cpu")
    args.update(kw)
    return DevicePagedKVCache(cfg, **args)


def test_default_head_map_is_the_reference_grouping():
    np.testing.assert_array_equal(default_q_head_to_kv_head(8, 2), [0, 0, 0, 0, 1, 1, 1, 1])
    with pytest.raises(ValueError):
        default_q_head_to_kv_head(6, 4)


def test_constructor_rejects_bad_head_counts():
    with pytest.raises(ValueError):
        _cache(num_attention_heads=6, num_key_value_heads=4)
    with pytest.raises(ValueError):
        _cache(num_attention_heads=34, num_key_value_heads=2)  # more than 16 query heads per KV head
    with pytest.raises(ValueError):
        _cache(batch_size=0)


def test_append_rejects_a_token_index_that_is_not_the_cached_length():
    c = _cache()
    rows = np.zeros((2, 1, 64), np.float32)
    with pytest.raises(ValueError, match="expected token_index 0"):
        c.append_step(0, rows, rows, 5)


def test_shapes_and_layers_are_checked():
    c = _cache()
    with pytest.raises(ValueError):
        c.append_step(0, np.zeros((3, 1, 64), np.float32), np.zeros((3, 1, 64), np.float32), 0)  # 3 KV heads
    with pytest.raises(ValueError):
        c.append_step(0, np.zeros((2, 1, 64), np.float32), np.zeros((2, 2, 64), np.float32), 0)  # token counts differ
    with pytest.raises(ValueError):
        c.ingest_prefill_cache(2, np.zeros((2, 4, 64), np.float32), np.zeros((2, 4, 64), np.float32))
    with pytest.raises(ValueError, match="no cached tokens"):
        c.decode_layer(1, np.zeros((4, 64), np.float32))
    with pytest.raises(ValueError):
        c.ingest_prefill_cache(0, np.zeros((2, 4, 64), np.float32), np.zeros((2, 4, 64), np.float32), context_length=3)


def test_block_cache_checks_before_device_work():
    from dotcache_amd.block_cache import DeviceVllmPagedKVCache

    cfg = DotCacheConfig(head_dim=32, group_size=32, tokens_per_page=4)
    with pytest.raises(ValueError, match="block_size"):
        DeviceVllmPagedKVCache(config=cfg, num_hidden_layers=1, num_attention_heads=4, num_key_value_heads=2,
                               block_size=8, device="cpu")
    c = DeviceVllmPagedKVCache(config=cfg, num_hidden_layers=1, num_attention_heads=4, num_key_value_heads=2,
                               block_size=4, device="cpu")
    rows = np.zeros((1, 2, 32), np.float32)
    with pytest.raises(ValueError, match="out of order"):
        c.write_slots(0, rows, rows, [7 * 4 + 2])  # offset 2 of an empty block
    with pytest.raises(ValueError):
        c.write_slots(0, rows, rows, [0, 1])  # one slot per row
    with pytest.raises(ValueError, match="unique"):
        c.sync_layer_blocks(0, np.zeros((2, 2, 4, 32)), np.zeros((2, 2, 4, 32)), block_ids=[3, 3])
    with pytest.raises(ValueError, match="no cached tokens"):
        c.decode_layer(0, np.zeros((4, 32), np.float32))
    with pytest.raises(ValueError, match="expected token_index 0"):
        c.append_step(0, np.zeros((2, 1, 32)), np.zeros((2, 1, 32)), 4)


def test_block_cache_keeps_live_rows_and_gives_their_store_back(monkeypatch):
    """The fp32 rows of live blocks follow them while the row store grows and
    shrinks, reach the final encode whole, and the store is given back with
    the blocks.  (The encode launches are replaced by what they store.)"""
    import torch

    from dotcache_amd.block_cache import DeviceVllmPagedKVCache
    from dotcache_amd.config import DotCacheConfig
    from dotcache_amd.page_pool import DevicePagePool

    P, H, hd, L = 4, 2, 32, 2
    final = []

    def rows_with(self, v_pool, k, v, kp, ks, vp, vs, *, keep=None):
        if keep is not None:
            at = np.flatnonzero(keep[2] >= 0)
            for buf, x in zip(keep[:2], (k, v)):
                buf[torch.from_numpy(keep[2][at])] = x[torch.from_numpy(at)].float()

    monkeypatch.setattr(DevicePagePool, "encode_rows_with", rows_with)
    monkeypatch.setattr(DevicePagePool, "encode_streams_with",
                        lambda self, v_pool, k, v, tables: final.append((k.clone(), v.clone(), tables.clone())))
    cache = DeviceVllmPagedKVCache(config=DotCacheConfig(head_dim=hd, tokens_per_page=P), num_hidden_layers=L,
                                   num_attention_heads=H, num_key_value_heads=H, block_size=P, device="cpu", reserve_blocks=2)
    rng = np.random.default_rng(7)
    held = [dict() for _ in range(L)]

    def check():
        for lid in range(L):
            live = {b: r for b, r in held[lid].items() if 0 < len(r) < P}
            assert set(cache._row_slots[lid]) == set(live)
            n = cache._row_store[lid].shape[0]
            assert n <= 4 * len(live) and sorted([*cache._row_slots[lid].values(), *cache._free_slots[lid]]) == list(range(n))
            for blk, rows in live.items():
                got = cache._row_store[lid][cache._row_slots[lid][blk]][:, :, : len(rows)]  # [2, H, t, hd]
                assert torch.equal(got, torch.stack(rows, dim=2)), (lid, blk)

    def write(lid, blocks, counts):
        slots = np.concatenate([b * P + len(held[lid].get(b, ())) % P + np.arange(c) for b, c in zip(blocks, counts)])
        kv = torch.from_numpy(rng.normal(size=(2, len(slots), H, hd)).astype(np.float32))
        final.clear()
        cache.write_slots(lid, kv[0], kv[1], slots)
        whole = []
        for i, s in enumerate(slots.tolist()):
            if s % P == 0:
                held[lid][s // P] = []
            held[lid][s // P].append(kv[:, i])
            if s % P == P - 1 and i >= P - 1 and slots[i - P + 1] == s - P + 1:
                whole.append(s // P)
        done = [b for b in blocks if len(held[lid][b]) == P and b not in whole]
        if done:  # one encode of the blocks that filled up, from their fp32 rows
            (k, v, tables), = final
            for i, b in enumerate(done):
                for x, kind, table in ((k, 0, tables[0]), (v, 1, tables[1])):
                    want = torch.stack([r[kind] for r in held[lid][b]], dim=1)
                    assert torch.equal(x[i * H:(i + 1) * H], want)
                    assert table[i * H:(i + 1) * H, 0].tolist() == cache._map["KV"[kind]][lid][b].tolist()
        else:
            assert not final
        check()

    for lid in range(L):
        write(lid, range(1), [1])
        write(lid, range(1, 40), [1 + b % 3 for b in range(39)])   # the store grows
        write(lid, range(36), [P - len(held[lid][b]) for b in range(36)])  # most blocks fill up: it shrinks
        assert cache._row_store[lid].shape[0] == 8
        write(lid, [36, 41, 37, 50], [1, 3, 1, P])
    # random writes: blocks taken up again, reused from their first slot, whole ones among them
    for _ in range(60):
        lid = int(rng.integers(L))
        blocks = rng.permutation(12)[: int(rng.integers(1, 12))]
        write(lid, blocks.tolist(), [int(rng.integers(1, P - len(held[lid].get(int(b), ())) % P + 1)) for b in blocks])
    cache.clear_layer(0)
    held[0].clear()
    check()
    assert cache._row_store[0].shape[0] == 0
    cache.clear()
    assert all(s.shape[0] == 0 for s in cache._row_store)
