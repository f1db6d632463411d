"""Which kernel a decode call runs on (dkv_decode_route): the host's rules over descriptors, without a GPU."""

import ctypes

import pytest

from dartkv_amd import _lib

F32, FP, BF = 0, 1, 2
NAMES = ("none", "pages", "tiles", "dense", "general")


def _page(D=128, tokens=128, key="uniform", bits=2, value_bits=None, kgroup=128, vgroup=64, promoted=0, at=1 << 20):
    s = _lib.Segment()
    s.tokens, s.key_group, s.value_group, s.promoted = tokens, kgroup, vgroup, promoted
    s.key_kind = _lib.KEY_MIXED if key == "dart" else _lib.KEY_UNIFORM
    s.value_kind, s.key_bits, s.value_bits = _lib.VALUE_UNIFORM, 0 if key == "dart" else bits, value_bits or bits
    for i in range(5):
        s.key[i], s.key_bh[i] = at, 1 << 12
    for i in range(3):
        s.value[i], s.value_bh[i] = at, 1 << 12
    return s


def _dense(tokens, at=1 << 20):
    s = _lib.Segment()
    s.tokens, s.key_kind, s.value_kind = tokens, _lib.KEY_DENSE, _lib.VALUE_DENSE
    s.key[0] = s.value[0] = at
    s.key_bh[0] = s.value_bh[0] = tokens * 128
    return s


def _args(segments, *, B=1, H=8, G=4, D=128, dtype=BF, q_dtype=None, meta=FP, tail=None, run=None, dense=0, splits=1):
    table = (_lib.Segment * max(1, len(segments)))(*segments)
    a = _lib.DecodeArgs(q_dtype=dtype if q_dtype is None else q_dtype, B=B, Hq=H * G, Hkv=H, D=D, cache_dtype=dtype,
                        meta_dtype=meta, n_segments=len(segments), segments_host=ctypes.addressof(table),
                        n_splits=splits, rest_dense_tokens=dense)
    if tail is not None:
        a.tail = tail
    if run is not None:
        first, count = run
        s = segments[first]
        a.fast_first, a.fast_count, a.fast_splits = first, count, count
        a.fast_promoted, a.fast_value_group = s.promoted, s.value_group
        a.fast_key_bits, a.fast_value_bits = s.key_bits, s.value_bits
    a._table = table  # (kept with the arguments)
    return a


def _route(a):
    k = _lib.decode_kernels(a)
    return NAMES[k.run], NAMES[k.rest]


@pytest.mark.parametrize("call,route", [
    (dict(), "tiles"),
    (dict(D=64), "tiles"),
    (dict(dtype=FP, G=16), "tiles"),
    (dict(D=96), "general"),
    (dict(G=17), "general"),
    (dict(dtype=F32), "general"),
    (dict(q_dtype=FP), "general"),
    (dict(meta=BF), "general"),
])
def test_rest_by_call(call, route):
    D = call.get("D", 128)
    assert _route(_args([_page(D=D, kgroup=64)] * 3, tail=_dense(40), **call)) == ("none", route)


@pytest.mark.parametrize("page,route", [
    (dict(kgroup=32), "tiles"), (dict(kgroup=384, tokens=300), "tiles"), (dict(key="dart", promoted=7), "tiles"),
    (dict(bits=8, vgroup=32), "tiles"), (dict(bits=4, vgroup=200), "tiles"),
    (dict(kgroup=48), "general"), (dict(kgroup=192), "general"), (dict(vgroup=16), "general"),
    (dict(bits=4, value_bits=2), "general"), (dict(key="dart", promoted=0), "general"),
    # sizes whose byte offsets would leave 32 bits (or 24, where they are factors)
    (dict(kgroup=1 << 16), "tiles"), (dict(kgroup=1 << 17), "general"), (dict(kgroup=1 << 27, bits=4), "general"),
    (dict(bits=8, vgroup=4096), "tiles"), (dict(bits=8, vgroup=1 << 15, tokens=1 << 16), "general"),
    (dict(tokens=1 << 16), "tiles"), (dict(tokens=(1 << 16) + 1), "general"),
])
def test_rest_by_page_layout(page, route):
    assert _route(_args([_page(**page)] * 2)) == ("none", route)


def test_rest_of_one_packed_run_of_one_layout():
    a, b, d = _page(), _page(kgroup=64), _dense(32)
    assert _route(_args([d, a, a, d], tail=_dense(5))) == ("none", "tiles")
    assert _route(_args([a, b])) == ("none", "general")
    assert _route(_args([a, d, a])) == ("none", "general")
    assert _route(_args([d], tail=_dense(200, at=8))) == ("none", "general")  # rows off 16 bytes
    assert _route(_args([d])) == ("none", "tiles")


def test_page_runs():
    d, dart16 = _dense(32), _page(key="dart", promoted=32, value_bits=2)
    for G in (1, 2, 4, 8):
        assert _route(_args([d] + [dart16] * 40, G=G, B=64, run=(1, 40), dense=32)) == ("pages", "dense")
    assert _route(_args([d] + [dart16] * 4, G=16, run=(1, 4), dense=32)) == ("tiles", "tiles")
    assert _route(_args([dart16] * 4, G=16, q_dtype=F32, run=(0, 4))) == ("tiles", "none")
    assert _route(_args([dart16] * 4 + [_page(key="dart", promoted=32, tokens=40)], run=(0, 4))) == ("pages", "tiles")
    other = _page(bits=4, value_bits=2)
    assert _route(_args([other] * 64, B=64, G=8, run=(0, 64))) == ("pages", "none")  # two code widths


def test_dense_entries_come_in_pieces():
    """Work items of the tile kernel: the packed segments, and 128-token pieces of the longest dense entry for each."""
    pages = [_page(kgroup=64)] * 5

    def units(a):
        return _lib.decode_kernels(a).rest_units
    assert units(_args(pages)) == 5
    assert units(_args([_dense(32)] + pages, tail=_dense(128))) == 5 + 2
    assert units(_args([_dense(32)] + pages, tail=_dense(129))) == 5 + 2 * 2
    assert units(_args([_dense(1 << 19)], tail=_dense(1))) == 2 * (1 << 12)
    assert units(_args([_dense(4000)] + pages, dtype=F32)) == 6  # the general kernel takes whole segments


@pytest.mark.parametrize("bits,dtype,G,pages,vgroup,run", [
    # eight rows: 2 and 4 bits always, 8 bits where the launch fills the device (2,048 pages of all heads)
    (2, BF, 8, 1, 64, "tiles"), (4, FP, 8, 1, 128, "tiles"), (8, BF, 8, 255, 64, "pages"), (8, FP, 8, 256, 64, "tiles"),
    (2, BF, 4, 255, 64, "pages"), (2, FP, 4, 256, 64, "tiles"), (2, BF, 2, 256, 64, "pages"), (2, BF, 1, 257, 128, "tiles"),
    (4, BF, 4, 2047, 64, "pages"), (4, BF, 4, 2048, 64, "tiles"), (4, BF, 2, 8191, 64, "pages"), (4, BF, 1, 8192, 128, "tiles"),
    (4, BF, 1, 256, 32, "tiles"), (4, BF, 1, 255, 32, "pages"),
    (4, FP, 4, 256, 64, "tiles"), (4, FP, 2, 256, 64, "pages"), (4, FP, 2, 257, 128, "tiles"),
    (4, FP, 1, 1023, 64, "pages"), (4, FP, 1, 1024, 64, "tiles"),
    (8, BF, 2, 256, 64, "tiles"), (8, BF, 1, 4095, 64, "pages"), (8, BF, 1, 4096, 64, "tiles"),
    (8, FP, 4, 384, 64, "tiles"), (8, FP, 4, 385, 64, "pages"), (8, FP, 1, 256, 64, "pages"),
    (2, BF, 8, 999, 16, "pages"),  # eight value groups: the page kernel only
])
def test_uniform_page_runs(bits, dtype, G, pages, vgroup, run):
    a = _args([_page(bits=bits, vgroup=vgroup)] * pages, B=1, H=8, G=G, dtype=dtype, run=(0, pages))
    assert _route(a) == (run, "none")
