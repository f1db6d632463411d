"""The one-launch read-back of a cache (dkv_materialize) against its segments dequantized one by one, bit for bit, over
its load forms (octets of 2-, 4- and 8-bit codes, Dart pages, dense pieces) and the element-wise form of every other
layout and type, at partial chunks."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
BF, FP, F32, F64 = torch.bfloat16, torch.float16, torch.float32, torch.float64


@pytest.mark.parametrize("T,D,dtype,cfg", [
    (1000, 128, BF, dict(promote_ratio=0.25, sink_tokens=32, hold_partial_pages=True)),
    (1001, 64, FP, dict(promote_ratio=0.3, key_group_size=64, value_group_size=32)),
    (517, 128, FP, dict(bits=4, key_group_size=32, sink_tokens=3, hold_partial_pages=True)),
    (300, 64, BF, dict(bits=8, value_group_size=24)),
    (256, 128, F32, dict(key_group_size=32, value_group_size=32, sink_tokens=2)),
    (700, 128, BF, dict(page_size=300, key_group_size=104, bits=4, sink_tokens=200)),   # chunks inside a page
    (130, 8, F32, dict(page_size=16, key_group_size=8, value_group_size=8, promote_ratio=0.25)),
    # element by element: group sizes that are not octets, other metadata, float64, an odd head_dim
    (90, 32, BF, dict(page_size=8, key_group_size=3, value_group_size=6, promote_ratio=0.25)),
    (200, 64, FP, dict(metadata_dtype=BF, bits=4)),
    (200, 64, F64, dict(metadata_dtype=F64, bits=2, promote_ratio=0.25)),
    (60, 20, F32, dict(page_size=16, key_group_size=8, value_group_size=8, bits=4)),
    (140, 64, BF, dict(local_tokens=4, page_size=32, key_group_size=32)),
])
def test_get_equals_the_segments(T, D, dtype, cfg):
    import dartkv_amd as dart
    from dartkv_amd.cache import _materialize
    g = torch.Generator().manual_seed(T)
    k, v = (torch.randn(2, 3, T, D, generator=g, dtype=F32).to(dtype).to(DEV) for _ in range(2))
    cache = dart.DartKVCache(dart.DartKVCacheConfig(**cfg))
    cache.append(k[..., :T - 1, :], v[..., :T - 1, :])
    cache.append(k[..., T - 1:, :], v[..., T - 1:, :])
    print("case", T, D, dtype, cfg, flush=True)
    segments = cache.iter_segments()
    keys = torch.cat([_materialize(ks) for ks, _ in segments], dim=-2)
    values = torch.cat([_materialize(vs) for _, vs in segments], dim=-2)
    got_k, got_v = cache.get()
    torch.cuda.synchronize()
    assert got_k.is_contiguous() and got_k.dtype == dtype and got_k.shape == (2, 3, T, D)
    bits = torch.int64 if dtype == F64 else torch.int32 if dtype == F32 else torch.int16
    assert torch.equal(got_k.view(bits), keys.contiguous().view(bits))
    assert torch.equal(got_v.view(bits), values.contiguous().view(bits))


def test_captured_get_outlives_the_descriptor_table():
    """A captured read-back keeps no pointer to the decode plan's table, which the next sealed page replaces: it replays
    over the pages themselves, which stay where they are while the pool has room."""
    import dartkv_amd as dart
    g = torch.Generator().manual_seed(2)
    k, v = (torch.randn(2, 2, 700, 128, generator=g).to(BF).to(DEV) for _ in range(2))
    cache = dart.DartKVCache(dart.DartKVCacheConfig(promote_ratio=0.25, hold_partial_pages=True))
    cache.append(k[..., :513, :], v[..., :513, :])
    cache.append(k[..., 513:550, :], v[..., 513:550, :])
    ref = [t.clone() for t in cache.get()]  # (the plan and its table are built)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        cache.get()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert cache._materialize_all() is None
        got = cache.get()
    for _ in range(3):
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, ref))

    def storage():
        return [t.data_ptr() for t in (cache._key_pool.tensors["low_values"], cache._value_pool.tensors["values"],
                                       cache._tail_key, cache._tail_value)]
    before, plan = storage(), cache.decode_plan(cache.device)
    cache.append(k[..., 550:645, :], v[..., 550:645, :])
    assert cache.decode_plan(cache.device) is not plan
    if storage() == before:
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a[..., :512, :], b[..., :512, :]) for a, b in zip(got, ref))


@pytest.mark.parametrize("T,table", [(90, False), (8191, False), (8192, True)])
def test_get_of_dense_pieces_alone(T, table):
    """Two copies for few elements, the one-launch kernel over a descriptor table for 2^20 and more."""
    import dartkv_amd as dart
    k = torch.randn(1, 2, T, 64, device=DEV).to(BF)
    cache = dart.DartKVCache(dart.DartKVCacheConfig(sink_tokens=32, page_size=10000, hold_partial_pages=True))
    cache.append(k, -k)
    got_k, got_v = cache.get()
    assert torch.equal(got_k, k) and torch.equal(got_v, -k) and got_k.data_ptr() != k.data_ptr()
    assert (cache._decode_plan_cache is not None) == table
