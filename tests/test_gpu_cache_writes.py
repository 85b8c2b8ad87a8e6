"""The caches' one-launch writes where they can go wrong: rows of several
blocks interleaved in one call, a block filled and reused in one call, rows
that fill a live block, 16-bit inputs, head_dims off the 8-channel lanes, and
the prompt ingest's tail.  Pages must equal the oracle's encode bit for bit."""
import numpy as np
import pytest

from oracle import dotcache_oracle as O
from tests.helpers import hard_values, pool_page_to_oracle

pytestmark = pytest.mark.gpu


def _same(page, want):
    for name in ("payload", "scales", "bias", "escape_payload"):
        a, b = getattr(page, name), getattr(want, name)
        assert (a is None) == (b is None), name
        if a is not None:
            assert np.array_equal(np.ascontiguousarray(a).view(np.uint8), np.ascontiguousarray(b).view(np.uint8)), name


def _oracle(rows, hd, gs, kind, mode):
    return O.encode_page(rows, head_dim=hd, group_size=gs, kind=kind, bits=4, mode=mode)


@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("hd,gs", [(64, 32), (96, 32), (30, 32)])
def test_interleaved_blocks_and_reuse(hd, gs, dtype):
    import torch

    from dotcache_amd.block_cache import DeviceVllmPagedKVCache
    from dotcache_amd.config import DotCacheConfig

    P, H = 16, 2
    print(f"block writes hd {hd} {dtype}", flush=True)
    cache = DeviceVllmPagedKVCache(config=DotCacheConfig(head_dim=hd, group_size=gs, tokens_per_page=P), num_hidden_layers=1,
                                   num_attention_heads=2 * H, num_key_value_heads=H, block_size=P, reserve_blocks=2)
    rng = np.random.default_rng(hd)
    held = {}

    def write(slots):
        x = torch.from_numpy(hard_values(rng, len(slots) * H, hd).reshape(len(slots), H, hd)).to(getattr(torch, dtype)).cuda()
        y = torch.from_numpy(hard_values(rng, len(slots) * H, hd).reshape(len(slots), H, hd)).to(getattr(torch, dtype)).cuda()
        cache.write_slots(0, x, y, np.asarray(slots))
        for i, s in enumerate(slots):
            if s % P == 0:
                held[s // P] = {}
            held[s // P][s % P] = (x[i].float().cpu().numpy(), y[i].float().cpu().numpy())

    def check():
        for blk, rows in held.items():
            for k, kind in enumerate(("K", "V")):
                for h in range(H):
                    e = cache.block_entry(0, h, blk, kind)
                    assert e.token_count == len(rows) and e.finalized == (len(rows) == P)
                    want = np.stack([rows[t][k][h] for t in range(len(rows))])
                    _same(e.page, _oracle(want, hd, gs, kind, "M0" if len(rows) == P else "M3"))

    write([0, 5 * P, 1, 5 * P + 1, 2])                        # two blocks, interleaved
    check()
    write(list(range(3, P)) + list(range(2 * P, 3 * P)))       # fills a live block; a whole block
    check()
    write(list(range(2 * P, 3 * P)) + list(range(2 * P, 2 * P + 3)))  # rewritten whole, then reused, in one call
    check()
    with pytest.raises(ValueError, match="out of order"):
        write([7 * P, 7 * P + 1, 5 * P + 9])
    assert cache.block_entry(0, 0, 7, "K").token_count == 2    # the rows before the error landed


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T", [1, 15, 16, 17, 100])
def test_prompt_ingest_and_append(T, dtype):
    import torch

    from dotcache_amd.config import DotCacheConfig
    from dotcache_amd.kv_cache import DevicePagedKVCache

    P, H, B, hd = 16, 2, 2, 64
    cache = DevicePagedKVCache(DotCacheConfig(head_dim=hd, tokens_per_page=P), num_hidden_layers=1, num_attention_heads=H,
                               num_key_value_heads=H, batch_size=B, reserve_pages_per_stream=1)
    rng = np.random.default_rng(T)
    n = T + 21
    kv = [torch.from_numpy(hard_values(rng, B * H * n, hd).reshape(B, H, n, hd)).to(getattr(torch, dtype)).cuda() for _ in "KV"]
    cache.ingest_prefill_cache(0, kv[0][:, :, :T], kv[1][:, :, :T])
    cache.append_step(0, kv[0][:, :, T:T + 1], kv[1][:, :, T:T + 1], T)
    cache.append_step(0, kv[0][:, :, T + 1:], kv[1][:, :, T + 1:], T + 1)
    for kind, x in zip("KV", kv):
        rows = x.float().cpu().numpy()
        pool = cache.k_pool if kind == "K" else cache.v_pool
        for b in range(B):
            for h in range(H):
                ids = cache.page_ids(0, b, h, kind)
                assert len(ids) == n // P
                for i, pid in enumerate(ids):
                    assert cache.page(0, b, h, i, kind).header.token_start == i * P
                    _same(pool_page_to_oracle(pool, pid, kind), _oracle(rows[b, h, i * P:(i + 1) * P], hd, 32, kind, "M0"))
                if n % P:
                    _same(pool_page_to_oracle(pool, cache.tail_page_id(0, b, h, kind), kind),
                          _oracle(rows[b, h, n // P * P:], hd, 32, kind, "M3"))
