"""The tile decode kernel (16-bit caches outside the page kernels' forms) against the oracle, at the edges of its
tiles and of its dispatch.

Its weights are fp32 (three 16-bit parts; in fp16 within three steps of 2^-37 of the largest) and its products exact,
so its error is that of fp32 logits and sums: a logit of size L carries about L 2^-24 (L below 50 here: 3e-6 relative
in its weight) and the sums over at most 1,700 tokens the same order, under the 1e-5 that fp32 caches are held to;
test_small_weights_keep_their_bits has the long sums.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
BF, FP = torch.bfloat16, torch.float16


def _rel_err(a, b):
    a, b = a.detach().float().cpu().flatten(2), b.detach().float().cpu().flatten(2)
    return float(((a - b).abs().amax(-1) / b.abs().amax(-1).clamp_min(1e-30)).max())


def _route(q, cache, **options):
    from dartkv_amd.attention import decode_route
    return decode_route(q.to(DEV), cache, **options)


def _run(B, Hkv, G, D, T, dtype, cfg, updates=(), n_splits=None, kernel="tiles"):
    import dartkv_amd as dart
    from dartkv_amd import synthetic
    from oracle import dart_oracle as O
    cfg = dict(dict(bits=2, page_size=128, key_group_size=128, value_group_size=64, sink_tokens=32,
                    hold_partial_pages=True, metadata_dtype=torch.float16), **cfg)
    k, v, q = synthetic.outlier_kv(B, Hkv, T, D, query_heads=Hkv * G, dtype=dtype, seed=7 + T + G, outliers=D // 16)
    oc, cache = O.OracleCache(O.OracleConfig(**cfg)), dart.DartKVCache(dart.DartKVCacheConfig(**cfg))
    start = 0
    for n in (*updates, T - sum(updates)):
        part = slice(start, start + n)
        oc.append(k[..., part, :], v[..., part, :])
        cache.append(k[..., part, :].to(DEV), v[..., part, :].to(DEV))
        start += n
    ref = O.streamed_attention(q, oc, return_fp32=True)[1]
    out = torch.empty(B, Hkv * G, D, dtype=torch.float32, device=DEV)
    print("case", B, Hkv, G, D, T, dtype, cfg, n_splits, flush=True)
    assert _route(q, cache, fast=False, n_splits=n_splits) == ("none", kernel)
    dart.decode_attention(q.to(DEV), cache, out_f32=out, fast=False, n_splits=n_splits)
    torch.cuda.synchronize()
    return _rel_err(out.unsqueeze(2), ref)


@pytest.mark.parametrize("G,D,T,dtype,cfg", [
    # head ratios: the padded rows of 4, 8 and 16, on Dart pages
    (1, 128, 700, BF, dict(promote_ratio=0.25)),
    (3, 128, 700, FP, dict(promote_ratio=0.25)),
    (5, 64, 700, BF, dict(promote_ratio=0.25)),
    (8, 128, 700, FP, dict(promote_ratio=0.25)),
    (9, 64, 700, FP, dict(promote_ratio=0.25)),
    (16, 128, 700, BF, dict(promote_ratio=0.25)),
    # promoted counts: one, not a multiple of 8 or 32, more than one block of 32, every channel
    (4, 128, 500, BF, dict(promote_ratio=0.008)),
    (4, 64, 500, FP, dict(promote_ratio=0.3)),
    (6, 128, 500, BF, dict(promote_ratio=0.3, key_group_size=64)),
    (4, 128, 500, FP, dict(promote_ratio=0.6, key_group_size=32)),
    (4, 128, 500, BF, dict(promote_ratio=1.0)),
    # code widths, key groups (several per tile, a padded one, one wider than the page), value groups
    (4, 128, 500, BF, dict(key_group_size=32, value_group_size=32)),
    (4, 64, 500, FP, dict(key_group_size=256, value_group_size=16)),
    (7, 128, 500, BF, dict(bits=4, key_group_size=64, value_group_size=48)),
    (2, 64, 500, BF, dict(bits=4, key_group_size=32, value_group_size=64)),
    # value rows of 42 and 18 bytes: off the shared loads' width
    (4, 128, 500, BF, dict(value_group_size=56)),
    (3, 128, 500, FP, dict(promote_ratio=0.25, value_group_size=56)),
    (4, 64, 500, BF, dict(value_group_size=24)),
    (4, 128, 500, FP, dict(bits=8, key_group_size=64, value_group_size=128)),
    (12, 64, 500, BF, dict(bits=8, key_group_size=32, value_group_size=32)),
    # segments that are not one full tile: short pages, pages of 256 tokens (two and four tiles), partial pages
    (4, 128, 333, BF, dict(page_size=40, key_group_size=32, promote_ratio=0.25)),
    (4, 128, 1200, FP, dict(page_size=256, key_group_size=128, promote_ratio=0.25)),
    (4, 64, 1200, BF, dict(page_size=256, key_group_size=64, bits=8)),
    (4, 128, 1000, BF, dict(hold_partial_pages=False, promote_ratio=0.25)),
    (3, 128, 1000, FP, dict(hold_partial_pages=False, bits=4, key_group_size=64)),
    (3, 64, 33, BF, dict(hold_partial_pages=False)),                 # one packed token
    # dense tokens only, none, and more than a tile of them
    (3, 64, 20, BF, {}),
    (9, 128, 160, FP, {}),
    (4, 64, 400, BF, dict(sink_tokens=0)),
    (4, 128, 900, BF, dict(sink_tokens=300, local_tokens=200, promote_ratio=0.25)),
])
def test_tile_kernel_vs_oracle(G, D, T, dtype, cfg):
    assert _run(2, 2, G, D, T, dtype, cfg) <= 1e-5


@pytest.mark.parametrize("G,D,T,dtype,cfg", [
    (4, 96, 400, BF, dict(key_group_size=64, value_group_size=32)),          # head_dim
    (4, 128, 400, torch.float32, dict(key_group_size=64)),                   # cache type
    (4, 128, 400, BF, dict(metadata_dtype=BF)),
    (4, 128, 400, FP, dict(page_size=80, key_group_size=40)),
    (4, 128, 400, FP, dict(value_group_size=16)),                            # eight value groups
    (4, 64, 400, BF, dict(bits=4, value_bits=2)),
])
def test_what_the_tile_kernel_leaves_to_the_general_kernel(G, D, T, dtype, cfg):
    assert _run(2, 2, G, D, T, dtype, cfg, kernel="general") <= 1e-5


@pytest.mark.parametrize("n_splits", [1, 2, 5, 64])
def test_tile_kernel_split_counts(n_splits):
    """Splits that hold several pages, a page and the dense pieces, or nothing but a dense piece."""
    assert _run(1, 2, 6, 128, 900, BF, dict(promote_ratio=0.25), n_splits=n_splits) <= 1e-5


def test_rest_of_a_page_run_takes_the_tile_kernel():
    """A short last page beside a run the page kernel takes: the run's records and the tile kernel's meet in one merge
    (the page kernel's bar, its weights are 16-bit)."""
    import dartkv_amd as dart
    from dartkv_amd import synthetic
    from oracle import dart_oracle as O
    cfg = dict(bits=2, page_size=128, key_group_size=128, value_group_size=64, sink_tokens=32, promote_ratio=0.25,
               hold_partial_pages=False, metadata_dtype=torch.float16)
    k, v, q = synthetic.outlier_kv(2, 4, 1000, 128, query_heads=16, dtype=BF, seed=3)
    oc, cache = O.OracleCache(O.OracleConfig(**cfg)), dart.DartKVCache(dart.DartKVCacheConfig(**cfg))
    oc.append(k, v)
    cache.append(k.to(DEV), v.to(DEV))
    ref = O.streamed_attention(q, oc, return_fp32=True)[1]
    out = torch.empty(2, 16, 128, dtype=torch.float32, device=DEV)
    assert _route(q, cache) == ("pages", "tiles")
    dart.decode_attention(q.to(DEV), cache, out_f32=out)
    torch.cuda.synchronize()
    assert _rel_err(out.unsqueeze(2), ref) <= 2e-3


@pytest.mark.parametrize("dtype", [BF, FP])
def test_tile_kernel_keeps_infinite_dense_values(dtype):
    """A dense tail token with an infinite value gives infinities where fp32 attention does, and no NaN from the
    positions past the tail."""
    import dartkv_amd as dart
    g = torch.Generator().manual_seed(1)
    k, v = (torch.randn(1, 2, 300, 64, generator=g).to(dtype) for _ in range(2))
    v[0, 1, 299, 5] = float("inf")
    q = torch.randn(1, 6, 1, 64, generator=g).to(dtype)
    cache = dart.DartKVCache(dart.DartKVCacheConfig(bits=4, page_size=128, key_group_size=64, value_group_size=64,
                                                    hold_partial_pages=True))
    cache.append(k.to(DEV), v.to(DEV))
    assert _route(q, cache) == ("none", "tiles")
    out = dart.fused_dart_attention(q.to(DEV), cache).cpu()
    torch.cuda.synchronize()
    expected = torch.zeros(1, 6, 1, 64, dtype=torch.bool)
    expected[0, 3:, 0, 5] = True
    assert torch.equal(torch.isinf(out), expected) and not torch.isnan(out).any()


@pytest.mark.parametrize("G,T,dtype,q_dtype,cfg", [
    (16, 700, BF, BF, dict(promote_ratio=0.25)),                 # sixteen rows on Dart pages, dense pieces beside
    (16, 900, FP, torch.float32, dict(promote_ratio=0.5)),       # a query of another type: three exact parts
    (16, 900, BF, FP, dict(promote_ratio=0.125, value_group_size=16)),
    (16, 1000, BF, torch.float64, dict(promote_ratio=0.25, hold_partial_pages=False)),  # a short page in the rest
    (8, 900, BF, BF, dict(bits=4, promote_ratio=0.0)),           # uniform pages with eight rows
    (8, 1000, FP, FP, dict(bits=8, promote_ratio=0.0, hold_partial_pages=False)),
    (8, 800, BF, FP, dict(bits=2, promote_ratio=0.0)),           # ... and another query type: the page kernel
    (8, 800, BF, BF, dict(bits=4, value_bits=2, promote_ratio=0.0)),
])
def test_page_runs_the_tile_kernel_takes(G, T, dtype, q_dtype, cfg):
    """Full-page runs on their way through the page path's arguments (splits, events, dense rest, records)."""
    import dartkv_amd as dart
    from dartkv_amd import synthetic
    from oracle import dart_oracle as O
    cfg = dict(dict(bits=2, page_size=128, key_group_size=128, value_group_size=64, sink_tokens=32,
                    hold_partial_pages=True, metadata_dtype=torch.float16), **cfg)
    k, v, q = synthetic.outlier_kv(2, 2, T, 128, query_heads=2 * G, dtype=torch.float32, seed=T + G)
    k, v, q = k.to(dtype), v.to(dtype), q.to(q_dtype)
    oc, cache = O.OracleCache(O.OracleConfig(**cfg)), dart.DartKVCache(dart.DartKVCacheConfig(**cfg))
    oc.append(k, v)
    cache.append(k.to(DEV), v.to(DEV))
    ref = O.streamed_attention(q, oc, return_fp32=True)[1]
    out = torch.empty(2, 2 * G, 128, dtype=torch.float32, device=DEV)
    print("case", G, T, dtype, q_dtype, cfg, flush=True)
    events = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    for e in events:
        e.record()
    got = dart.decode_attention(q.to(DEV), cache, out_f32=out, fast=True, fast_events=events)
    torch.cuda.synchronize()
    assert got.dtype == q_dtype and events[0].elapsed_time(events[1]) >= 0
    tiles = G == 16 or (q_dtype == dtype and "value_bits" not in cfg and cfg["bits"] < 8)
    rest = "tiles" if q_dtype == dtype else "general"
    if cfg["hold_partial_pages"]:
        rest = "tiles" if tiles else "dense"
    assert _route(q, cache, fast=True) == ("tiles" if tiles else "pages", rest)
    assert _rel_err(out.unsqueeze(2), ref) <= (1e-5 if tiles else 2e-3)


@pytest.mark.parametrize("G,Q,D,dtype,q_dtype,launches,cfg", [
    (4, 4, 64, BF, BF, 1, dict(promote_ratio=0.25)),                 # no page run: sixteen rows in one launch
    (3, 5, 128, FP, FP, 1, dict(key_group_size=64)),
    (6, 3, 128, BF, BF, 2, dict(key_group_size=64, promote_ratio=0.25)),  # twelve rows, then six
    (4, 3, 128, BF, BF, 1, dict(bits=4)),                            # page runs: rows the page kernels do not have
    (2, 8, 128, FP, FP, 1, dict(bits=8)),
    (1, 3, 128, BF, BF, 1, dict(promote_ratio=0.25)),
    (16, 2, 128, BF, BF, 2, dict(bits=4)),
    (4, 3, 128, BF, FP, 2, dict(promote_ratio=0.25)),                # pages only the page kernel takes: 8 + 4 rows
    (4, 3, 128, BF, BF, 2, dict(bits=4, value_group_size=16)),
    (4, 3, 128, FP, FP, 2, dict(bits=4, value_bits=2)),
    (4, 3, 128, BF, BF, 2, dict(bits=4, value_local_tokens=70)),     # ... beside pages with a dense value window
    (4, 4, 64, torch.float32, torch.float32, 1, dict(bits=4)),       # the general kernel
])
def test_query_tokens_share_launches(G, Q, D, dtype, q_dtype, launches, cfg, monkeypatch):
    import dartkv_amd as dart
    from dartkv_amd import attention, synthetic
    from oracle import dart_oracle as O
    cfg = dict(dict(bits=2, page_size=128, key_group_size=128, value_group_size=64, sink_tokens=32,
                    hold_partial_pages=True, metadata_dtype=torch.float16), **cfg)
    k, v, _ = synthetic.outlier_kv(2, 2, 700, D, query_heads=2, dtype=torch.float32, seed=G + Q)
    q = torch.randn(2, Q, 2 * G, D, generator=torch.Generator().manual_seed(Q)).to(q_dtype).transpose(1, 2)
    k, v = k.to(dtype), v.to(dtype)
    oc, cache = O.OracleCache(O.OracleConfig(**cfg)), dart.DartKVCache(dart.DartKVCacheConfig(**cfg))
    oc.append(k, v)
    cache.append(k.to(DEV), v.to(DEV))
    ref = O.streamed_attention(q, oc, return_fp32=True)[1]
    print("case", G, Q, D, dtype, q_dtype, cfg, flush=True)
    calls, decode = [], attention.decode_attention
    monkeypatch.setattr(attention, "decode_attention", lambda *a, **kw: calls.append(0) or decode(*a, **kw))
    plain = torch.empty(2, 2 * G, Q, D, dtype=torch.float32, device=DEV)
    strided = torch.empty(2, Q, 2 * G, D, dtype=torch.float32, device=DEV).transpose(1, 2)
    for out in (plain, strided):
        got = attention._multi_token_attention(q.to(DEV), cache, out_f32=out)
        torch.cuda.synchronize()
        assert got.shape == out.shape and got.dtype == q_dtype and got.is_contiguous()
        assert torch.equal(got.float(), out.to(q_dtype).float())
        assert _rel_err(out, ref) <= (1e-5 if launches == 1 or G in (6, 16) else 2e-3)
    assert len(calls) == 2 * launches


@pytest.mark.parametrize("D,pages,dtype", [
    (128, 24, BF), (128, 33, BF), (64, 64, FP), (128, 300, BF),  # one record per page: the first, and past a thread's 32
    (192, 40, torch.float32), (96, 30, BF), (256, 130, FP),      # thread groups that do not fill the workgroup
])
def test_merge_of_many_records(D, pages, dtype):
    """One record per page, weights over many orders of magnitude and records of masked-out size."""
    import dartkv_amd as dart
    from oracle import dart_oracle as O
    g = torch.Generator().manual_seed(pages + D)
    T = 8 * pages
    k, v, q = (torch.randn(1, 2, n, D, generator=g).to(dtype) for n in (T, T, 3))
    k[:, :, : T // 2] *= 4.0
    q = q.reshape(1, 6, 1, D)
    cfg = dict(bits=4, page_size=8, key_group_size=8, value_group_size=32)
    oc, cache = O.OracleCache(O.OracleConfig(**cfg)), dart.DartKVCache(dart.DartKVCacheConfig(**cfg))
    oc.append(k, v)
    cache.append(k.to(DEV), v.to(DEV))
    ref = O.streamed_attention(q, oc, return_fp32=True)[1]
    out = torch.empty(1, 6, D, dtype=torch.float32, device=DEV)
    print("case", D, pages, dtype, flush=True)
    dart.decode_attention(q.to(DEV), cache, out_f32=out, n_splits=pages)
    assert _rel_err(out.unsqueeze(2), ref) <= 2e-5  # logits to about 100: 100 x 2^-24 relative in a weight


@pytest.mark.parametrize("dtype,pad,skip", [(BF, 1, 0), (FP, 8, 4), (BF, 8, 0), (FP, 0, 1)])
def test_query_alignment(dtype, pad, skip):
    """Queries whose heads or base are off 16 bytes take the narrow loads, the same bits as a contiguous query."""
    import dartkv_amd as dart
    g = torch.Generator().manual_seed(3)
    k, v = (torch.randn(2, 2, 300, 64, generator=g).to(dtype).to("cuda") for _ in range(2))
    cache = dart.DartKVCache(dart.DartKVCacheConfig(promote_ratio=0.25, hold_partial_pages=True))
    cache.append(k, v)
    q = torch.randn(2, 6, 1, 64, generator=g).to(dtype).to("cuda")
    flat = torch.zeros(skip + 2 * 6 * (64 + pad), dtype=dtype, device="cuda")
    strided = flat[skip:].view(2, 6, 1, 64 + pad)[..., :64]
    strided.copy_(q)
    assert torch.equal(dart.decode_attention(strided, cache), dart.decode_attention(q, cache))


def _peaked(G, D, T, dtype, gap):
    """A cache whose first token holds almost all of the softmax weight of every query head, and a query: the other
    tokens' logits lie ``gap`` to ``gap`` + 6 below.  Values are positive."""
    import dartkv_amd as dart
    g = torch.Generator().manual_seed(T + G)
    k = 0.1 * torch.randn(1, 2, T, D, generator=g)
    k[..., 0] = -torch.randint(0, 2, (T,), generator=g).float()  # two values: the codes keep them
    k[:, :, 0, 0] = gap / 6.0
    v = 0.5 + torch.rand(1, 2, T, D, generator=g)
    q = 0.1 * torch.randn(1, 2 * G, 1, D, generator=g)
    q[..., 0] = 6.0
    cache = dart.DartKVCache(dart.DartKVCacheConfig(bits=2, page_size=128, key_group_size=64, value_group_size=32,
                                                    hold_partial_pages=True))
    return cache, k.to(dtype), v.to(dtype), q.to(dtype)


@pytest.mark.parametrize("gap", [14.0, 18.0, 24.0])  # weights of 2^-20 to 2^-43
@pytest.mark.parametrize("G,D,dtype", [(3, 64, FP), (7, 128, FP), (12, 64, FP), (16, 128, FP), (3, 64, BF), (12, 128, BF)])
def test_small_weights_keep_their_bits(G, D, dtype, gap):
    """8,191 negligible tokens in one split against 64 bits.  The split's 64 tiles are added to the result and to the sum
    of the weights one by one, 2^-24 relative each at most: 128 x 2^-24 = 7.6e-6; fp16 weights add 2e-7, and fp32
    logits 30 x 2^-24 of the 2^-7 that the negligible tokens hold."""
    import dartkv_amd as dart
    cache, k, v, q = _peaked(G, D, 8192, dtype, gap)
    cache.append(k.to(DEV), v.to(DEV))
    dk, dv = (t.cpu().double() for t in cache.get())
    logits = torch.matmul(q.double().view(1, 2, G, D), dk.transpose(-1, -2))
    ref = torch.matmul(torch.softmax(logits, -1), dv).view(1, 2 * G, 1, D)
    out = torch.empty(1, 2 * G, D, dtype=torch.float32, device=DEV)
    print("case", G, D, dtype, gap, flush=True)
    assert _route(q, cache, fast=False, n_splits=1) == ("none", "tiles")
    dart.decode_attention(q.to(DEV), cache, scale=1.0, out_f32=out, fast=False, n_splits=1)
    got = out.cpu().double().view(1, 2 * G, 1, D)
    assert float(((got - ref).abs() / ref.abs()).max()) <= 7.8e-6


@pytest.mark.parametrize("G,dtype", [(3, FP), (7, FP), (12, FP), (3, BF), (7, BF), (12, BF)])
def test_infinite_value_of_a_small_weight(G, dtype):
    """A held token with a weight of about 2^-50 and an infinite value gives an infinity, as fp32 weights do."""
    import dartkv_amd as dart
    cache, k, v, q = _peaked(G, 64, 300, dtype, 32.0)
    v[0, 1, 299, 5] = float("inf")
    cache.append(k.to(DEV), v.to(DEV))
    print("case", G, dtype, flush=True)
    assert _route(q, cache, fast=False, n_splits=1) == ("none", "tiles")
    out = dart.decode_attention(q.to(DEV), cache, scale=1.0, fast=False, n_splits=1).cpu()
    expected = torch.zeros(1, 2 * G, 1, 64, dtype=torch.bool)
    expected[0, G:, 0, 5] = True
    assert torch.equal(torch.isinf(out), expected) and not torch.isnan(out).any()


@pytest.mark.parametrize("dtype,q_dtype", [(BF, torch.float32), (FP, torch.float32), (BF, FP)])
def test_infinite_key_under_a_query_of_another_type(dtype, q_dtype):
    """Sixteen rows on Dart pages, a held token with an infinite key channel whose query elements are short and
    negative: its logit is minus infinity, its weight zero, and nothing is NaN."""
    import dartkv_amd as dart
    g = torch.Generator().manual_seed(5)
    k, v = (torch.randn(1, 2, 300, 128, generator=g).to(dtype) for _ in range(2))
    k[0, :, 299, 3] = float("inf")
    q = torch.randn(1, 32, 1, 128, generator=g)
    q[..., 3] = -0.5
    q = q.to(q_dtype)
    cache = dart.DartKVCache(dart.DartKVCacheConfig(promote_ratio=0.25, key_group_size=128, value_group_size=64,
                                                    hold_partial_pages=True))
    cache.append(k.to(DEV), v.to(DEV))
    dk, dv = (t.cpu().double() for t in cache.get())
    logits = torch.matmul(q.double().view(1, 2, 16, 128), dk.transpose(-1, -2)) / 128 ** 0.5
    ref = torch.matmul(torch.softmax(logits, -1), dv).view(1, 32, 1, 128)
    out = torch.empty(1, 32, 128, dtype=torch.float32, device=DEV)
    print("case", dtype, q_dtype, flush=True)
    assert _route(q, cache) == ("tiles", "tiles")
    dart.decode_attention(q.to(DEV), cache, out_f32=out)
    assert _rel_err(out.unsqueeze(2), ref) <= 1e-5


@pytest.mark.parametrize("G,T,dtype,n_splits,fast,cfg", [
    (6, 1400, BF, None, None, dict(promote_ratio=0.25, sink_tokens=300, local_tokens=500)),
    (6, 1400, FP, 3, None, dict(promote_ratio=0.25, sink_tokens=129, local_tokens=257)),   # pieces of one token
    (3, 1000, FP, 64, False, dict(key_group_size=64, local_tokens=700)),
    (4, 900, BF, None, False, dict(key_group_size=64, sink_tokens=900)),                   # dense pieces only
    (16, 1700, BF, None, True, dict(promote_ratio=0.25, local_tokens=600)),                # beside a page run
    (16, 1700, FP, 2, True, dict(promote_ratio=0.25, local_tokens=600, sink_tokens=256)),
    (8, 1700, BF, None, True, dict(bits=4, local_tokens=600)),
    (8, 1700, FP, 5, True, dict(bits=2, local_tokens=384, sink_tokens=0)),
])
def test_long_dense_windows_in_pieces(G, T, dtype, n_splits, fast, cfg):
    import dartkv_amd as dart
    from dartkv_amd import synthetic
    from oracle import dart_oracle as O
    cfg = dict(dict(bits=2, page_size=128, key_group_size=128, value_group_size=64, sink_tokens=32,
                    hold_partial_pages=True, metadata_dtype=torch.float16), **cfg)
    k, v, q = synthetic.outlier_kv(2, 2, T, 128, query_heads=2 * G, dtype=dtype, seed=T + G)
    oc, cache = O.OracleCache(O.OracleConfig(**cfg)), dart.DartKVCache(dart.DartKVCacheConfig(**cfg))
    oc.append(k, v)
    cache.append(k.to(DEV), v.to(DEV))
    ref = O.streamed_attention(q, oc, return_fp32=True)[1]
    out = torch.empty(2, 2 * G, 128, dtype=torch.float32, device=DEV)
    print("case", G, T, dtype, n_splits, fast, cfg, flush=True)
    run, rest = _route(q, cache, n_splits=n_splits, fast=fast)
    assert rest == "tiles" and run == ("tiles" if fast else "none")
    dart.decode_attention(q.to(DEV), cache, out_f32=out, n_splits=n_splits, fast=fast)
    assert _rel_err(out.unsqueeze(2), ref) <= 1e-5


@pytest.mark.parametrize("dtype", [BF, FP])
@pytest.mark.parametrize("n_splits", [None, 1, 40])
def test_logits_of_minus_infinity(dtype, n_splits):
    """Tokens with a logit of minus infinity have no weight, also where they are a whole piece and split of their own;
    where every token is one, the result is NaN."""
    import dartkv_amd as dart
    g = torch.Generator().manual_seed(9)
    k, v = (torch.randn(1, 2, 260, 64, generator=g).to(dtype) for _ in range(2))
    q = torch.randn(1, 6, 1, 64, generator=g).to(dtype)
    q[..., 7] = 1.0
    k[..., 256:, 7] = float("-inf")
    cfg = dict(bits=2, page_size=128, key_group_size=64, value_group_size=32, sink_tokens=400, hold_partial_pages=True)
    for first in (0, 256):
        cache = dart.DartKVCache(dart.DartKVCacheConfig(**cfg))
        cache.append(k[..., first:, :].to(DEV), v[..., first:, :].to(DEV))
        assert _route(q, cache, n_splits=n_splits) == ("none", "tiles")
        print("case", dtype, n_splits, first, flush=True)
        got = dart.decode_attention(q.to(DEV), cache, n_splits=n_splits).cpu().double()
        logits = torch.matmul(q.double().view(1, 2, 3, 64), k[..., first:, :].double().transpose(-1, -2)) / 8.0
        ref = torch.matmul(torch.softmax(logits, -1), v[..., first:, :].double()).view(1, 6, 1, 64)
        if first:
            assert torch.isnan(ref).all() and torch.isnan(got).all()
        else:
            assert float((got - ref).norm() / ref.norm()) <= (4e-3 if dtype == BF else 5e-4)  # the output's rounding


@pytest.mark.parametrize("dtype,q_dtype,cfg,kernel,splits", [
    (BF, BF, dict(key_group_size=64), "tiles", 16),
    (BF, torch.float32, dict(key_group_size=64), "general", 32),
    (BF, BF, dict(key_group_size=64, metadata_dtype=BF), "general", 32),
    (FP, FP, dict(page_size=80, key_group_size=40), "general", 32),
    (FP, FP, dict(key_group_size=64, sink_tokens=4000), "tiles", 16),  # pieces of one dense segment
])
def test_split_counts_of_the_kernel_that_runs(dtype, q_dtype, cfg, kernel, splits):
    """2,048 waves of the tile kernel, 4,096 workgroups of the general kernel (128 batch-head pairs)."""
    import dartkv_amd as dart
    k = torch.randn(16, 8, 4000, 64, device=DEV).to(dtype)
    cache = dart.DartKVCache(dart.DartKVCacheConfig(bits=2, value_group_size=32, hold_partial_pages=True, **cfg))
    cache.append(k, k)
    q = torch.randn(16, 8, 1, 64, device=DEV).to(q_dtype)
    assert _route(q, cache) == ("none", kernel)
    dart.decode_attention(q, cache)
    (template, _), = cache.decode_plan(q.device).call_layouts.values()
    assert template.n_splits == splits
