"""Keys quantized along tokens from registers (groups of 32, 64 and 128; uniform and Dart pages) and the eight-element dequantize kernel,
bit for bit against the oracle: every code width and source type, tokens that do not fill a group, a block or a page,
strided sources, and the non-finite report."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
BF, FP, F32 = torch.bfloat16, torch.float16, torch.float32


def _same(a, b):
    a, b = a.cpu().contiguous(), b.contiguous()
    return a.dtype == b.dtype and a.shape == b.shape and torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def _data(shape, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(shape, generator=g)
    x[..., ::16] *= 10.0
    return x.to(dtype)


@pytest.mark.parametrize("shape,dtype,bits,group,meta", [
    ((2, 3, 256, 128), BF, 2, 64, FP),
    ((1, 2, 300, 64), FP, 4, 32, FP),      # a block of 44 tokens, its last group padded
    ((3, 200, 128), F32, 8, 128, F32),
    ((2, 1, 33, 64), BF, 8, 32, BF),
    ((1, 1, 129, 192), FP, 2, 128, FP),    # one token past a block; three row pieces
    ((2, 2, 1, 64), F32, 4, 64, FP),
    ((130, 64), BF, 4, 128, None),
    ((2, 2, 100, 96), BF, 4, 64, FP),      # rows that are not whole pieces: the copy form
    ((2, 2, 100, 128), BF, 4, 40, FP),
])
def test_quantize_along_tokens_vs_oracle(shape, dtype, bits, group, meta):
    import dartkv_amd as dart
    from oracle import dart_oracle as O
    x = _data(shape, dtype, sum(shape) + bits)
    print("case", shape, dtype, bits, group, meta, flush=True)
    got = dart.quantize(x.to(DEV), bits=bits, group_size=group, metadata_dtype=meta, axis=-2)
    ref = O.quantize(x, bits=bits, group_size=group, metadata_dtype=meta, axis=-2)
    for name in ("values", "scale", "zero_point"):
        assert _same(getattr(got, name), getattr(ref, name)), name
    assert _same(got.dequantize(), ref.dequantize())
    for out in (F32, BF, FP):
        assert _same(got.dequantize(dtype=out), ref.dequantize(dtype=out)), out


@pytest.mark.parametrize("D,dtype,cfg", [
    (128, BF, dict(bits=2, key_group_size=64, hold_partial_pages=True)),
    (64, FP, dict(bits=4, key_group_size=128, sink_tokens=5)),             # a short last page
    (64, F32, dict(bits=8, key_group_size=32, page_size=96)),
    (128, F32, dict(bits=2, key_group_size=32, value_group_size=32, sink_tokens=2)),
    (128, FP, dict(bits=2, key_group_size=128, page_size=256)),            # two blocks per page
])
def test_uniform_pages_vs_oracle_from_a_strided_source(D, dtype, cfg):
    """Keys and values as a projection leaves them, [B, T, heads, D] seen as [B, heads, T, D]."""
    import dartkv_amd as dart
    from oracle import dart_oracle as O
    k, v = (_data((2, 523, 3, D), dtype, s).transpose(1, 2) for s in (1, 2))
    oc, cache = O.OracleCache(O.OracleConfig(**cfg)), dart.DartKVCache(dart.DartKVCacheConfig(**cfg))
    oc.append(k, v)
    cache.append(k.to(DEV), v.to(DEV))
    print("case", D, dtype, cfg, flush=True)
    pairs = list(zip(cache.iter_segments(), oc.segments()))
    assert len(pairs) == len(oc.segments()) == len(cache.iter_segments())
    for got, ref in pairs:
        for g, r in zip(got, ref):
            if isinstance(g, torch.Tensor):
                assert _same(g, r)
            else:
                assert all(_same(getattr(g, n), getattr(r, n)) for n in ("values", "scale", "zero_point"))


@pytest.mark.parametrize("D,dtype,ratio,cfg", [
    (64, BF, 0.25, dict(key_group_size=128)),                              # last page of 11 tokens: half a page each
    (64, FP, 0.25, dict(key_group_size=32, sink_tokens=73)),               # 66 tokens
    (64, FP, 0.5, dict(key_group_size=64, channel_selection="variance")),
    (128, BF, 0.25, dict(key_group_size=64, channel_selection="variance", sink_tokens=73)),
    (128, BF, 0.125, dict(key_group_size=32, page_size=100)),
    (128, FP, 0.25, dict(key_group_size=64, page_size=16)),
    (128, F32, 0.25, dict(key_group_size=128, channel_selection="variance")),
    (96, F32, 0.25, dict(key_group_size=32, sink_tokens=60)),
    (64, BF, 1.0, dict(key_group_size=64)),                                # every channel promoted
])
def test_dart_pages_vs_oracle_from_a_strided_source(D, dtype, ratio, cfg):
    """Scores (both selections), the chosen channels in their order, low and high codes, scales and zero points."""
    import dartkv_amd as dart
    from oracle import dart_oracle as O
    cfg = dict(cfg, bits=2, value_group_size=32, promote_ratio=ratio)
    k, v = (_data((2, 523, 3, D), dtype, s).transpose(1, 2) for s in (3, 4))
    oc, cache = O.OracleCache(O.OracleConfig(**cfg)), dart.DartKVCache(dart.DartKVCacheConfig(**cfg))
    oc.append(k, v)
    cache.append(k.to(DEV), v.to(DEV))
    print("case", D, dtype, ratio, cfg, flush=True)
    pairs = [(g, r) for g, r in zip(cache.iter_segments(), oc.segments()) if not isinstance(g[0], torch.Tensor)]
    assert len(pairs) == (523 - cfg.get("sink_tokens", 0) + cfg.get("page_size", 128) - 1) // cfg.get("page_size", 128)
    for (got, _), (ref, _) in pairs:
        for name in ("low_values", "high_values", "channel_indices", "scale", "zero_point"):
            assert _same(getattr(got, name), getattr(ref, name)), name


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("axis", [-1, -2])
def test_quantize_rejects_non_finite_values(bad, axis):
    import dartkv_amd as dart
    x = _data((2, 2, 130, 64), BF, 3)
    x[1, 1, 129, 63] = bad
    with pytest.raises(ValueError, match="finite"):
        dart.quantize(x.to(DEV), bits=4, group_size=64, axis=axis)
    x[1, 1, 129, 63] = 0.0
    dart.quantize(x.to(DEV), bits=4, group_size=64, axis=axis)  # the report is cleared


def test_non_finite_input_is_reported_before_a_bad_metadata_type():
    """The reference's order of checks (non-finite values first, src/dart/quantization.py:159-160): both faults at once raise ValueError."""
    import dartkv_amd as dart
    x = torch.ones(4, 64, device="cuda")
    x[1, 3] = float("nan")
    with pytest.raises(ValueError, match="finite"):
        dart.quantize(x, bits=4, group_size=32, metadata_dtype=torch.int8)
    with pytest.raises(TypeError, match="metadata dtype"):
        dart.quantize(torch.ones(4, 64, device="cuda"), bits=4, group_size=32, metadata_dtype=torch.int8)
    with pytest.raises(ValueError, match="finite"):
        dart.quantize(x, bits=4, group_size=32)
