"""Several query tokens over an F32 cache through the several-token kernel
(kraken-infer_amd/csrc/attention_rows_f32.hip) at its edges: both head sizes, every group
size, a last row group that is not full, splits that only the later tokens reach,
one token's rows alone in a group, an odd number of row groups, cache layers.

Against the oracle (double accumulation): f32 sums of at most 128 products and of the
weighted values, outputs below 4 in size: 4e-6 absolute is 16 units of f32's last
place at 2, where these shapes show 1e-6; an f16 operand anywhere misses by 1e-4."""
import numpy as np
import pytest

import kraken_hip as kh
import oracle


def inputs(seed, tokens, cap, heads, kv_heads, d, layers=1):
    rng = np.random.default_rng(seed)
    q = rng.standard_normal(tokens * heads * d).astype(np.float32)
    k, v = (rng.standard_normal(layers * cap * kv_heads * d).astype(np.float32) for _ in range(2))
    return q, k, v


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,start,heads,kv_heads,d", [
    (512, 0, 16, 8, 128),     # a prefill chunk: one split, 64 row groups
    (129, 900, 8, 8, 128),    # G = 1, the last group holds one token
    (37, 2100, 8, 2, 128),    # G = 4, splits
    (100, 0, 16, 8, 128), (101, 30, 16, 8, 128),
    (127, 0, 16, 8, 128), (128, 0, 16, 8, 128),   # either side of the rule
    (31, 737, 16, 8, 128), (32, 735, 16, 8, 128),  # and of its line for short contexts
    (90, 700, 8, 1, 128),     # G = 8, fewer splits than XCDs
    (21, 3000, 16, 2, 128),   # G = 8, two tokens per group, the last one alone
    (2, 70000, 4, 2, 128),    # a quarter of one group over many splits
    (175, 800, 4, 4, 64), (97, 601, 8, 1, 64),
])
def test_rows_f32_against_oracle(hip_ctx, monkeypatch, tokens, start, heads, kv_heads, d):
    print(f"rows f32 tokens={tokens} start={start} heads={heads}/{kv_heads} d={d}", flush=True)
    cap = start + tokens + 2
    q, k, v = inputs(tokens, tokens, cap, heads, kv_heads, d, layers=2)
    ops = kh.NumpyOps(hip_ctx)
    args = (q, k, v, 1, start, tokens, cap, heads, kv_heads, d)
    got = ops.attention_batched(*args)
    np.testing.assert_allclose(got, oracle.attention_batched(*args), rtol=0, atol=4e-6)
    monkeypatch.setenv("KRAKEN_DECODE_KERNEL", "vector")
    one = ops.attention_batched(*args)
    np.testing.assert_allclose(got, one, rtol=0, atol=8e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_rows_f32_later_tokens_values_do_not_leak(hip_ctx, monkeypatch, bad):
    tokens, start, heads, kv_heads, d = 70, 500, 16, 8, 128
    cap = start + tokens
    print(f"rows f32 {bad} in later value rows", flush=True)
    q, k, v = inputs(7, tokens, cap, heads, kv_heads, d)
    vr = v.reshape(cap, kv_heads, d)
    vr[start + 13, 0, 17] = bad
    vr[start + 64, 7, 127] = bad
    ops = kh.NumpyOps(hip_ctx)
    args = (q, k, v, 0, start, tokens, cap, heads, kv_heads, d)
    got = ops.attention_batched(*args).reshape(tokens, heads, d)
    assert np.isfinite(got[:13]).all() and np.isfinite(got[13:64, 2:]).all()
    assert not np.isfinite(got[13:, :2, 17]).any() and not np.isfinite(got[64:, 14:, 127]).any()
    monkeypatch.setenv("KRAKEN_DECODE_KERNEL", "vector")
    one = ops.attention_batched(*args).reshape(tokens, heads, d)
    finite = np.isfinite(one)
    np.testing.assert_array_equal(np.isfinite(got), finite)
    np.testing.assert_allclose(got[finite], one[finite], rtol=0, atol=8e-6)
