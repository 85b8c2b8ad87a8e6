"""Host-side rules that batched calls share with page-by-page ones: merge
windows and page bookkeeping, over the forms they accept (no GPU)."""
import numpy as np
import pytest

from dotcache_amd import _lib
from dotcache_amd.decode import merge_windows
from dotcache_amd.page_pool import DevicePagePool, PoolGeometry


def _pool(cap=64, hd=64):
    return DevicePagePool(PoolGeometry(hd, 32, cap), device="cpu", reserve_bytes=1 << 16, reserve_pages=16)


def _windows_by_sequence(pool, vpool, kt, vt, seq_pages):
    """The rule stated one sequence at a time."""
    f16 = _lib.FMT_M3_F16
    out = []
    for b, n in enumerate(seq_pages):
        exact = [[pool.formats_of(kt[b, h, p]) == f16 and vpool.formats_of(vt[b, h, p]) == f16 for p in range(n)]
                 for h in range(kt.shape[1])]
        if any(e != exact[0] for e in exact):
            return None
        begin = n
        while begin > 0 and exact[0][begin - 1]:
            begin -= 1
        tokens = max(sum(int(pool.tokens_of(kt[b, h, p])) for p in range(begin, n)) for h in range(kt.shape[1]))
        if begin < n and (begin == 0 or n - begin > 8 or tokens > 256):
            return None
        out.append((begin, n))
    return np.asarray(out) if any(b < n for b, n in out) else None


@pytest.mark.parametrize("seed", range(40))
def test_merge_windows_match_the_rule_per_sequence(seed):
    rng = np.random.default_rng(seed)
    B, H, S = int(rng.integers(1, 5)), int(rng.integers(1, 4)), int(rng.integers(1, 14))
    k, v = _pool(), _pool()
    seq = rng.integers(1, S + 1, size=B)
    kt, vt = (np.zeros((B, H, S), dtype=np.int32) for _ in range(2))
    for b in range(B):
        run = int(rng.integers(0, min(10, seq[b]) + 1)) * int(rng.random() < 0.8)
        for p in range(S):
            exact = seq[b] - run <= p < seq[b]
            tokens = int(rng.integers(1, 65)) if rng.random() < 0.5 else 64
            for h in range(H):
                fmt = (_lib.FMT_M3_F16, 0) if exact != (rng.random() < 0.01) else (_lib.FMT_M0_AFFINE, 4)
                kt[b, h, p] = k.allocate(*fmt, tokens=tokens)[0]
                vt[b, h, p] = v.allocate(*fmt, tokens=tokens)[0]
    got, want = merge_windows(k, v, kt, vt, seq), _windows_by_sequence(k, v, kt, vt, seq)
    assert (got is None) == (want is None)
    if want is not None:
        np.testing.assert_array_equal(got, want)


def test_pool_reuses_blobs_and_ids_in_order():
    pool = _pool()
    a = pool.allocate(_lib.FMT_M0_AFFINE, 4, 3, tokens=64)
    b = pool.allocate(_lib.FMT_M3_F16, 0, 2, tokens=1)
    starts = pool.descs_of(a)["block"].tolist()
    pool.free([a[0], b[0], a[2]])
    with pytest.raises(RuntimeError, match="not live"):
        pool.free([a[1], a[0]])
    assert pool.formats_of([a[1]])[0] == _lib.FMT_M0_AFFINE  # nothing was freed
    with pytest.raises(RuntimeError):
        pool.free([a[1], a[1]])
    c = pool.allocate(_lib.FMT_M0_AFFINE, 4, 3, tokens=2)
    assert c.tolist() == [a[0], b[0], a[2]]                       # ids oldest freed first
    assert pool.descs_of(c)["block"].tolist()[:2] == [starts[2], starts[0]]  # blobs last freed first
    assert pool.format_mask_of(c) == _lib.format_bit(_lib.FMT_M0_AFFINE, 4)
    many = pool.allocate(_lib.FMT_M0_SYMMETRIC, 8, 40, tokens=3)  # past the reserved descriptors
    assert len(set(many.tolist())) == 40 and (pool.tokens_of(many) == 3).all()


def test_a_negative_page_count_is_refused():
    pool = _pool()
    a = pool.allocate(_lib.FMT_M0_AFFINE, 4, 2, tokens=64)
    pool.free(a[:1])
    with pytest.raises(ValueError):
        pool.allocate(_lib.FMT_M0_AFFINE, 4, -1)
    assert pool.n_pages == 2 and pool.allocate(_lib.FMT_M0_AFFINE, 4, 0).size == 0


def test_deferred_headers_are_made_once_and_follow_token_counts():
    from dotcache_amd.config import DotCacheConfig
    from dotcache_amd.encode import make_header, resolve_encode_spec

    pool, cfg = _pool(), DotCacheConfig(head_dim=64)
    ids = pool.allocate(_lib.FMT_M0_AFFINE, 4, 3, tokens=64).tolist()
    template = make_header(cfg, resolve_encode_spec(cfg, kind="K"), kind="K", layer_id=0, kv_head_id=0, token_start=0, token_count=64)
    pool.headers.fill(ids, template, [0, 64, 128])
    assert len(pool.headers) == 3 and ids[1] in pool.headers
    assert pool.headers[ids[1]] is pool.headers.get(ids[1]) and pool.headers[ids[1]].token_start == 64
    pool.set_tokens(ids[2], 7)
    assert pool.headers[ids[2]].token_count == 7 and pool.headers[ids[0]].token_count == 64
    pool.free(ids[0])
    assert ids[0] not in pool.headers and sorted(pool.headers) == ids[1:]
    with pytest.raises(KeyError):
        pool.headers[ids[0]]
    # the rest of what a mapping does, on deferred entries too
    pool.headers.fill(ids[:1], template, [32])
    assert pool.headers.setdefault(ids[0], None).token_start == 32 and dict(pool.headers) == pool.headers
    pool.headers.fill(ids[:1], template, [32])
    del pool.headers[ids[0]]
    assert ids[0] not in pool.headers and pool.headers.pop(ids[0], None) is None
    pool.headers.fill(ids[:1], template, [32])
    pool.headers.clear()
    assert not pool.headers and list(pool.headers) == []


def test_headers_are_a_whole_dict_of_headers():
    """copy, |, reversed, popitem and the order of a dict, on deferred entries
    too; reading one moves nothing."""
    import copy
    import pickle

    from dotcache_amd.config import DotCacheConfig
    from dotcache_amd.encode import make_header, resolve_encode_spec

    pool, cfg = _pool(), DotCacheConfig(head_dim=64)
    template = make_header(cfg, resolve_encode_spec(cfg, kind="K"), kind="K", layer_id=0, kv_head_id=0, token_start=0, token_count=64)
    ids = pool.allocate(_lib.FMT_M0_AFFINE, 4, 4, tokens=64).tolist()
    h = pool.headers
    h.fill(ids[:3], template, [0, 64, 128])
    h[ids[3]] = template
    assert h[ids[2]].token_start == 128 and list(h) == ids and list(reversed(h)) == ids[::-1]
    want = h.copy()
    assert type(want) is dict and want == h and list(want) == ids and want[ids[1]] is h[ids[1]]
    assert [p for p in h if h[p].token_start >= 64] == ids[1:3]  # (making entries while iterating)
    assert h | {99: template} == {**want, 99: template} and {99: template} | h == {99: template, **want}
    assert repr(h) == repr(want) and copy.deepcopy(h) == want and pickle.loads(pickle.dumps(h)) == want
    assert h.popitem() == (ids[3], template)
    h |= {7: template}
    assert pool.headers is h and h.pop(7) is template and len(h) == 3
    h.clear()
    with pytest.raises(KeyError):
        h.popitem()


def test_uploaded_headers_are_page_headers_of_their_own():
    """Whatever carries the header of an uploaded page, the pool holds a
    PageHeader with its fields that is not the page's own."""
    from dataclasses import asdict
    from types import SimpleNamespace

    from dotcache_amd.config import DotCacheConfig
    from dotcache_amd.encode import make_header, resolve_encode_spec
    from dotcache_amd.types import EncodedPage, PageHeader

    cfg = DotCacheConfig(head_dim=64)
    spec = resolve_encode_spec(cfg, kind="K", mode="M3")
    plain = make_header(cfg, spec, kind="K", layer_id=3, kv_head_id=1, token_start=64, token_count=2)
    duck = SimpleNamespace(**asdict(plain))
    duck.to_dict = lambda: asdict(plain)
    pool = _pool()
    for header in (plain, duck):
        pid = int(pool.upload_pages([EncodedPage(header=header, escape_payload=np.zeros((2, 64), np.float16))])[0])
        assert type(pool.headers[pid]) is PageHeader and pool.headers[pid] == plain and pool.headers[pid] is not plain


def test_merge_windows_ignore_entries_past_the_pages():
    k, v = _pool(), _pool()
    ids = [p.allocate(_lib.FMT_M0_AFFINE, 4, 2, tokens=64) for p in (k, v)]
    tail = [p.allocate(_lib.FMT_M3_F16, 0, 1, tokens=9) for p in (k, v)]
    kt, vt = (np.array([[[*i.tolist(), *t.tolist(), 10**6, -7]]]) for i, t in zip(ids, tail))
    assert merge_windows(k, v, kt, vt, [3]).tolist() == [[2, 3]]


@pytest.mark.parametrize("whole", [0, 8192, 40])
def test_device_descriptors_follow_the_host_table(whole, monkeypatch):
    """Both uploads of changed descriptors (by index past ``WHOLE_TABLE_PAGES``
    pages, the whole table up to it) and the growth of the table."""
    from dotcache_amd import page_pool

    monkeypatch.setattr(page_pool, "WHOLE_TABLE_PAGES", whole)
    pool = _pool()
    rng = np.random.default_rng(whole)
    live: list[int] = []

    def check():
        n = pool.n_pages
        got = pool.device_descs()[:n].numpy().view(page_pool.DESC_DTYPE)
        np.testing.assert_array_equal(got, pool.descs_of(np.arange(n)))
        assert got["tokens"][live].min(initial=1) > 0

    for _ in range(30):
        new = pool.allocate(*((_lib.FMT_M3_F16, 0), (_lib.FMT_M0_AFFINE, 4))[int(rng.integers(2))], int(rng.integers(1, 9)), tokens=5)
        live += new.tolist()
        check()
        pool.set_tokens(rng.choice(live, size=min(3, len(live)), replace=False), int(rng.integers(1, 65)))
        check()
        gone = rng.choice(live, size=len(live) // 5, replace=False).tolist()
        pool.free(gone)
        live = [p for p in live if p not in gone]
        check()
    assert pool.n_pages > 16  # past the table reserved at first
