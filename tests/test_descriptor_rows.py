"""The descriptor table made run by run (CPU): the same bytes as one descriptor at a time, and the page run and dense
rest found on the arrays as by walking the entries, over sinks, breaks in the slots and rows, short pages, pools of
their own and unaligned blocks."""

import pytest
import torch

import dartkv_amd as dart
from dartkv_amd import _lib, cache as C
from dartkv_amd.pool import PagePool, PoolKeys, PoolMixedKey, PoolValues

CPU = torch.device("cpu")


def _pools(B, H, D, n, mixed, meta):
    if mixed:
        K = D // 4
        keys = {"low_values": ((0, B, H, D, 1, 32), torch.uint8), "high_values": ((0, B, H, K, 1, 32), torch.uint8),
                "channel_indices": ((0, B, H, K), torch.int32), "scale": ((0, B, H, D, 1), meta),
                "zero_point": ((0, B, H, D, 1), meta)}
    else:
        keys = {"values": ((0, B, H, D, 32), torch.uint8), "scale": ((0, B, H, D, 1), meta),
                "zero_point": ((0, B, H, D, 1), meta)}
    values = {"values": ((B, H, 0, D // 4), torch.uint8), "scale": ((B, H, 0, D // 64), meta),
              "zero_point": ((B, H, 0, D // 64), meta)}
    kpool, vpool = PagePool(keys, 0, 1, CPU), PagePool(values, 2, 0, CPU, align=64)
    kpool.reserve(n)
    vpool.reserve(n * 128)
    return kpool, vpool


def _cache(layout, mixed=True, B=2, H=3, D=128, meta=torch.float16, dtype=torch.bfloat16):
    """``layout``: ("d", tokens) dense, ("p", slot, first value row, tokens) a page."""
    cfg = dart.DartKVCacheConfig(bits=2, page_size=128, key_group_size=128, value_group_size=64, metadata_dtype=meta,
                                 promote_ratio=0.25 if mixed else 0.0, hold_partial_pages=True)
    cache = dart.DartKVCache(cfg)
    cache._shape, cache._dtype, cache._device = (B, H, D), dtype, CPU
    kpool, vpool = cache._key_pool, cache._value_pool = _pools(B, H, D, 24, mixed, meta)
    own, _ = _pools(B, H, D, 4, mixed, meta)  # a page pool of another launch
    for kind, *x in layout:
        if kind == "d":
            cache._keys.append(torch.zeros(B, H, x[0], D, dtype=dtype))
            cache._values.append(torch.zeros(B, H, x[0], D, dtype=dtype))
            continue
        slot, row, tokens = x
        pool = own if kind == "o" else kpool
        cache._keys.append(PoolMixedKey(pool, slot, tokens, D, 128, 128, 4, dtype) if mixed
                           else PoolKeys(pool, slot, tokens, D, 128, 128, 128, 2, dtype))
        cache._values.append(PoolValues(vpool, row, tokens, D, 128, D, 64, 2, dtype))
    return cache


def _walked_run(cache, descs, count):
    """The longest run of page-kernel entries and the dense rest, entry by entry."""
    mixed = cache.config.promote_ratio > 0

    def page(d):
        fields = [(d.key[i], d.key_bh[i], s) for i, s in (((0, 1), (1, 1), (2, 4), (3, 2), (4, 2)) if mixed
                                                         else ((0, 1), (3, 2), (4, 2)))]
        fields += [(d.value[i], d.value_bh[i], s) for i, s in ((0, 1), (1, 2), (2, 2))]
        return (d.tokens == 128 and d.key_kind == (_lib.KEY_MIXED if mixed else _lib.KEY_UNIFORM)
                and d.value_kind == _lib.VALUE_UNIFORM and all(a % 16 == 0 and bh * s % 16 == 0 for a, bh, s in fields))

    ok = [page(descs[i]) for i in range(count)]
    first, best, start = 0, 0, 0
    for i in range(count + 1):
        if i == count or not ok[i]:
            if i - start > best:
                first, best = start, i - start
            start = i + 1
    rest = [descs[i] for i in range(count) if not first <= i < first + best]
    dense = -1 if not all(C._dense16_ok(d) for d in rest) else max((d.tokens for d in rest), default=0)
    return (first if best else 0, best), dense


PAGES = [("p", i, 128 * i, 128) for i in range(6)]


@pytest.mark.parametrize("layout", [
    [("d", 32)] + PAGES,
    PAGES,
    [("d", 32)],
    [("d", 32)] + PAGES[:3] + [("p", 9, 384, 128), ("p", 10, 512, 128)] + [("d", 5)],    # a break in the slots
    PAGES[:2] + [("p", 2, 640, 128), ("p", 3, 768, 128), ("p", 4, 896, 128)],            # a break in the rows
    PAGES[:4] + [("p", 4, 512, 77)],                                                     # a short page
    PAGES[:2] + [("o", 2, 256, 128), ("o", 3, 384, 128), ("p", 4, 512, 128)],            # pages of another pool
    [("p", 0, 3, 128), ("p", 1, 131, 128)],                                              # value rows off 16 bytes
    [("p", 3, 384, 128), ("p", 2, 256, 128)],                                            # slots that go down
])
@pytest.mark.parametrize("mixed", [True, False])
def test_table_equals_one_descriptor_at_a_time(layout, mixed):
    cache = _cache(layout, mixed)
    plan = cache.decode_plan(CPU)
    pairs, keep = cache._sealed_pairs(), []
    ref = (_lib.Segment * len(pairs))()
    for desc, (kseg, vseg) in zip(ref, pairs):
        C.fill_segment(desc, kseg, vseg, keep)
    assert bytes(plan.host_table) == bytes(ref) == bytes(plan.table.numpy())
    run, dense = _walked_run(cache, ref, len(pairs))
    assert (plan.fast_first, plan.fast_count) == run and plan.rest_dense == dense
    assert plan.n_tokens == sum(C._segment_tokens(k) for k, _ in pairs)


def test_no_page_run_outside_the_page_kernels_layout():
    for kw in (dict(meta=torch.float32), dict(dtype=torch.float32), dict(D=64)):
        plan = _cache([("d", 32)] + PAGES, **kw).decode_plan(CPU)
        assert plan.fast_count == 0
