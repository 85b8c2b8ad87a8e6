"""``dc_score_pages`` / ``dc_mix_pages`` over every page format and the sizes
where their tiles end: token counts around 64, page capacities below and
above it, head_dims that are one or several 16-channel slices or no multiple
of 16, and query counts around a block's 4."""
import numpy as np
import pytest

from oracle import dotcache_oracle as O
from tests.helpers import hard_values, to_product_page

pytestmark = pytest.mark.gpu

FORMATS = [dict(bits=2), dict(bits=3), dict(bits=3, scheme="symmetric"), dict(bits=4), dict(bits=4, scheme="symmetric"),
           dict(bits=8), dict(bits=8, scheme="symmetric"), dict(mode="M3"), dict(mode="M3", escape_dtype="float32"),
           dict(mode="M3", escape_dtype="int8")]


def _groups(rng, hd, gs, fmt, lens, tpp, kind, layout):
    pages = [O.encode_pages(hard_values(rng, n, hd), tokens_per_page=tpp, head_dim=hd, group_size=gs, kind=kind,
                            layout=layout, **fmt) for n in lens]
    return pages, [[to_product_page(p) for p in g] for g in pages]


@pytest.mark.parametrize("fmt", FORMATS, ids=lambda f: "-".join(str(v) for v in f.values()))
@pytest.mark.parametrize("hd,gs,tpp,Q,lens,layout", [
    (128, 32, 64, 1, [1], "group_major"),
    (128, 32, 64, 3, [63, 63], "group_major"),
    (64, 16, 32, 4, [97, 97, 97], "group_major"),
    (96, 32, 100, 5, [257, 257], "token_major"),
    (256, 64, 128, 9, [700], "group_major"),
    (80, 48, 64, 2, [130], "group_major"),
    (48, 24, 64, 2, [70], "group_major"),
])
def test_grouped_logits_weights_and_output(fmt, hd, gs, tpp, Q, lens, layout):
    from dotcache_amd.backends import decode_grouped_multiquery_step_prepared_hip_tensor as grouped

    print(f"grouped {fmt} hd {hd} gs {gs} page {tpp} Q {Q} {lens} {layout}", flush=True)
    rng = np.random.default_rng(hd + tpp + Q)
    q = (rng.normal(size=(len(lens), Q, hd)) / np.sqrt(hd)).astype(np.float32)
    okp, kp = _groups(rng, hd, gs, fmt, lens, tpp, "K", layout)
    ovp, vp = _groups(rng, hd, gs, fmt, lens, tpp, "V", layout)
    logits, weights, out = (t.cpu().numpy() for t in grouped(list(q), kp, vp))
    for g in range(len(lens)):
        want = O.decode_multi_query_step(q[g], okp[g], ovp[g])
        # fp32 sums of up to 256 products of |q| < 0.5 and |k| < 60 (logits),
        # of 700 weights that sum to 1 and |v| < 60 (output): both orders stay
        # within n 2^-24 of the summed magnitudes, under 1e-4
        np.testing.assert_allclose(logits[g], want[0], atol=1e-4, rtol=1e-5)
        np.testing.assert_allclose(weights[g], want[1], atol=1e-5, rtol=1e-4)
        np.testing.assert_allclose(out[g], want[2], atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("kfmt,vfmt", [(FORMATS[i], FORMATS[(3 * i + 1) % len(FORMATS)]) for i in range(len(FORMATS))]
                         + [(dict(bits=4), dict(mode="M3", escape_dtype="int8"))],
                         ids=lambda f: "-".join(str(v) for v in f.values()))
@pytest.mark.parametrize("hd,gs,vgs,tpp,Q,layout", [
    (128, 32, 32, 64, 4, "group_major"),
    (96, 32, 64, 96, 2, "group_major"),
    (64, 16, 16, 32, 5, "token_major"),
    (256, 64, 32, 256, 16, "group_major"),
    (80, 16, 48, 100, 9, "group_major"),
    (160, 32, 32, 64, 1, "token_major"),
])
def test_tile_decode_matches_oracle(kfmt, vfmt, hd, gs, vgs, tpp, Q, layout):
    """The tile decode over every pair of formats: token counts of one unit, a
    partial unit, and several units per wave; one item per group and items of
    two pages that split a group.  The value pool also holds a 3-bit page that
    is not read, which keeps the MFMA kernel off the call."""
    from dotcache_amd import _lib
    from dotcache_amd.backends import clear_prepared_pools, prepare_pages_hip
    from dotcache_amd.backends import decode_grouped_multiquery_step_prepared_hip_tensor_output_only as fused
    from dotcache_amd.decode import set_decode_path

    print(f"tiles {kfmt} {vfmt} hd {hd} gs {gs}/{vgs} page {tpp} Q {Q} {layout}", flush=True)
    rng = np.random.default_rng(hd + tpp + Q)
    lens = [1, 64, tpp + 17, 5 * tpp - 3]
    q = (rng.normal(size=(len(lens), Q, hd)) / np.sqrt(hd)).astype(np.float32)
    okp, kp = _groups(rng, hd, gs, kfmt, lens, tpp, "K", layout)
    ovp, vp = _groups(rng, hd, vgs, vfmt, lens, tpp, "V", layout)
    want = O.decode_grouped(q, okp, ovp)
    clear_prepared_pools()
    kp, vp = ([prepare_pages_hip(g) for g in pages] for pages in (kp, vp))
    for pool in {id(g[0].pool): g[0].pool for g in vp}.values():
        pool.allocate(_lib.FMT_M0_AFFINE, 3)
    set_decode_path("mfma")
    try:
        with pytest.raises(ValueError, match="MFMA kernel does not cover"):
            fused(list(q), kp, vp)
        seen = {}
        for path in ("auto", "generic"):  # the tile kernel, and the generic kernel on the same pages
            set_decode_path(path)
            for pps in (None, 2, 100):
                seen[path] = got = fused(list(q), kp, vp, pages_per_split=pps).cpu().numpy()
                # fp32 products and sums on both sides, |out| < 60
                assert np.max(np.abs(got - want)) < 1e-4, f"{path}, pages per split {pps}"
        # two kernels: their sums run in different orders and round differently somewhere
        assert not np.array_equal(seen["auto"], seen["generic"])
    finally:
        set_decode_path("auto")
        clear_prepared_pools()


@pytest.mark.parametrize("kfmt,vfmt", [(FORMATS[i], FORMATS[(3 * i + 1) % len(FORMATS)]) for i in range(len(FORMATS))],
                         ids=lambda f: "-".join(str(v) for v in f.values()))
@pytest.mark.parametrize("hd,gs,vgs,tpp,Q,layout", [
    (48, 24, 24, 64, 4, "group_major"),
    (40, 20, 40, 32, 3, "token_major"),
    (30, 32, 32, 64, 1, "group_major"),   # one padded group, rows off 16 bytes
    (250, 50, 25, 96, 16, "group_major"),
])
def test_generic_decode_matches_oracle(kfmt, vfmt, hd, gs, vgs, tpp, Q, layout):
    """Geometries that 16-channel chunks do not tile have the generic kernel
    only."""
    from dotcache_amd.backends import clear_prepared_pools
    from dotcache_amd.backends import decode_grouped_multiquery_step_prepared_hip_tensor_output_only as fused

    print(f"generic {kfmt} {vfmt} hd {hd} gs {gs}/{vgs} page {tpp} Q {Q} {layout}", flush=True)
    rng = np.random.default_rng(hd + tpp + Q)
    lens = [1, 64, tpp + 17, 5 * tpp - 3]
    q = (rng.normal(size=(len(lens), Q, hd)) / np.sqrt(hd)).astype(np.float32)
    okp, kp = _groups(rng, hd, gs, kfmt, lens, tpp, "K", layout)
    ovp, vp = _groups(rng, hd, vgs, vfmt, lens, tpp, "V", layout)
    want = O.decode_grouped(q, okp, ovp)
    clear_prepared_pools()
    for pps in (None, 2):
        got = fused(list(q), kp, vp, pages_per_split=pps).cpu().numpy()
        # fp32 products and sums on both sides, |out| < 60
        assert np.max(np.abs(got - want)) < 1e-4, f"pages per split {pps}"


@pytest.mark.parametrize("Q", [8, 9, 16])
def test_decode_around_the_tiles_lds_limit(Q):
    """8-bit affine values in 16 groups of 16: 135 KiB of tiles for 8 query
    heads, 151 KiB for 9 to 16, which the generic kernel takes."""
    from dotcache_amd.backends import clear_prepared_pools
    from dotcache_amd.backends import decode_grouped_multiquery_step_prepared_hip_tensor_output_only as fused

    print(f"lds limit Q {Q}", flush=True)
    rng = np.random.default_rng(Q)
    lens, hd, tpp = [1, 97, 400], 256, 64
    q = (rng.normal(size=(len(lens), Q, hd)) / np.sqrt(hd)).astype(np.float32)
    okp, kp = _groups(rng, hd, 16, dict(bits=4), lens, tpp, "K", "group_major")
    ovp, vp = _groups(rng, hd, 16, dict(bits=8), lens, tpp, "V", "group_major")
    clear_prepared_pools()
    got = fused(list(q), kp, vp).cpu().numpy()
    assert np.max(np.abs(got - O.decode_grouped(q, okp, ovp))) < 1e-4


def test_mix_keeps_infinities_of_valid_rows_only():
    """An infinite value row makes its channels infinite, not NaN, also as a
    page's last token."""
    from dotcache_amd import attention_runtime as rt

    rng = np.random.default_rng(3)
    v = rng.normal(size=(37, 64)).astype(np.float32)
    v[36, 5] = np.inf
    page = to_product_page(O.encode_page(v, head_dim=64, group_size=32, kind="V", mode="M3", escape_dtype="float32"))
    w = np.full(37, 1 / 37, dtype=np.float32)
    got = rt.mix_page(w, page, backend="hip_mi355x")
    assert np.isposinf(got[5]) and np.isfinite(np.delete(got, 5)).all()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 256, 257, 1024, 1025, 2048, 2049, 7168, 7169, 8192, 8193, 20000])
def test_softmax_rows_in_place_and_out_of_place(n):
    """Around the block sizes' lines (256, 1024, 2048 and 7168 columns), a
    row's register columns (8 x 1024) and past them."""
    import ctypes as C

    import torch

    from dotcache_amd import _lib

    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    x = torch.randn((3, n + 5), generator=gen, device="cuda") * 4
    want = torch.softmax(x[:, :n].double(), dim=-1)
    y = torch.full((3, n), -1.0, device="cuda")
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    keep = x.clone()
    assert _lib.lib().dc_softmax_rows_to(x.data_ptr(), n + 5, y.data_ptr(), n, 3, n, stream) == 0
    assert torch.equal(x, keep)
    # each weight: one exp (2 ulp), a sum of n terms in a tree of depth < 32, one division
    assert float(((y - want).abs() / want).max()) < 40 * 2.0 ** -24 + 2e-7 * float((x - x.amax(-1, True)).abs().max())
    assert _lib.lib().dc_softmax_rows(x.data_ptr(), 3, n, n + 5, stream) == 0
    assert torch.equal(x[:, :n], y) and torch.equal(x[:, n:], keep[:, n:])


def test_softmax_of_many_short_rows_keeps_its_block_small():
    """4096 rows of 64 columns take less than three times 64 rows (blocks of
    1024 threads took seven times as long): both are one round of blocks."""
    import ctypes as C

    import torch

    from dotcache_amd import _lib

    x = torch.randn((4096, 64), device="cuda")
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)

    def us(rows):
        times = []
        for _ in range(20):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                assert _lib.lib().dc_softmax_rows(x.data_ptr(), rows, 64, 64, stream) == 0
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 50)
        return sorted(times)[len(times) // 2]

    us(64)
    assert us(4096) < 3 * us(64)
