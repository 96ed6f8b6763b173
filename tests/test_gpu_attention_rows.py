"""Several query tokens of one sequence through the several-token decode kernel
(kraken-infer_amd/csrc/attention_rows.hip) at its edges: a last row group that is
not full, one workgroup's rows from tokens with different causal limits, splits
that only the later tokens reach, each group size, cache layers, no split (in the
allocation-free entry's limit and forced), and a query scale at which an f16 query
would miss the bound.

Against the oracle with the f32 query: the tolerance of the decode kernels at that
query scale (test_gpu_attention.py, test_decode_keeps_f32_query_precision: 4e-6 at
unit scale and 2e-5 at 8x, above the split form's 2^-21 and below what an f16 query
shows).  The kernel that takes one workgroup per token is within the same bound."""
import importlib

import numpy as np
import pytest

import kraken_hip as kh
import oracle

D = 256


def inputs(seed, tokens, start, cap, heads, kv_heads, layers=1, scale=1.0):
    rng = np.random.default_rng(seed)
    q = (scale * rng.standard_normal(tokens * heads * D)).astype(np.float32)
    k, v = (rng.standard_normal(layers * cap * kv_heads * D).astype(np.float16).view(np.uint16)
            for _ in range(2))
    return q, k, v


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,start,heads,kv_heads,scale", [
    (2, 16400, 8, 2, 1.0),     # half of one row group, the most splits
    (5, 9000, 8, 2, 8.0),      # one row past a group of 16
    (17, 5000, 4, 4, 1.0),     # G = 1: 16 tokens per group, one token past it
    (33, 4100, 8, 4, 1.0),     # G = 2
    (63, 1300, 8, 2, 8.0),     # the most tokens before flash
    (63, 700, 4, 2, 1.0),      # the shortest context at two KV heads
    (25, 2100, 12, 3, 1.0),    # a grid that is no multiple of the eight XCDs
    (11, 5000, 2, 1, 1.0),     # one KV head
])
def test_rows_against_oracle(hip_ctx, monkeypatch, tokens, start, heads, kv_heads, scale):
    print(f"rows tokens={tokens} start={start} heads={heads}/{kv_heads}", flush=True)
    cap = start + tokens + 3
    q, k, v = inputs(tokens, tokens, start, cap, heads, kv_heads, layers=2, scale=scale)
    ops = kh.NumpyOps(hip_ctx)
    gate = np.random.default_rng(1).standard_normal(q.size).astype(np.float32)
    want = oracle.sigmoid_gate_mul(
        oracle.attention_batched(q, k, v, 1, start, tokens, cap, heads, kv_heads, D), gate)
    tol = 4e-6 if scale == 1.0 else 2e-5
    got = ops.attention_batched(q, k, v, 1, start, tokens, cap, heads, kv_heads, D, gate=gate)
    np.testing.assert_allclose(got, want, rtol=0, atol=tol)
    monkeypatch.setenv("KRAKEN_DECODE_KERNEL", "short")
    one = ops.attention_batched(q, k, v, 1, start, tokens, cap, heads, kv_heads, D, gate=gate)
    np.testing.assert_allclose(got, one, rtol=0, atol=2 * tol)


@pytest.mark.gpu
@pytest.mark.parametrize("keys_per_split", ["1", "37", "100000"])
def test_rows_at_any_split(hip_ctx, monkeypatch, keys_per_split):
    """One key per split is raised to the most splits of the merge; 37 keys give a
    last tile of five; 100000 one split, whose workgroup writes the output."""
    tokens, start, heads, kv_heads = 20, 4100, 8, 2
    print(f"rows keys per split {keys_per_split}", flush=True)
    monkeypatch.setenv("KRAKEN_DECODE_KEYS_PER_SPLIT", keys_per_split)
    cap = start + tokens
    q, k, v = inputs(3, tokens, start, cap, heads, kv_heads)
    got = kh.NumpyOps(hip_ctx).attention_batched(q, k, v, 0, start, tokens, cap, heads, kv_heads,
                                                 D)
    want = oracle.attention_batched(q, k, v, 0, start, tokens, cap, heads, kv_heads, D)
    np.testing.assert_allclose(got, want, rtol=0, atol=4e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv_heads,tokens", [(8, 2, 63), (16, 4, 40)])
def test_rows_fit_the_allocation_free_entry(hip_ctx, heads, kv_heads, tokens):
    """The plan keeps its partials within the allocation-free entry's array, so that
    entry takes the same shapes and gives the same bits."""
    start = 7000
    cap = start + tokens
    print(f"rows no-alloc {heads}/{kv_heads} tokens={tokens}", flush=True)
    q, k, v = inputs(5, tokens, start, cap, heads, kv_heads)
    bufs = [hip_ctx.buffer(x) for x in (q, k, v, np.zeros_like(q))]
    outs = []
    for name in ("attention_f32_batched_f16_kv_gated",
                 "attention_f32_batched_f16_kv_gated_no_alloc"):
        out = hip_ctx.buffer(byte_size=4 * q.size)
        hip_ctx.call(name, *bufs, 0, start, tokens, cap, heads, kv_heads, D, out)
        outs.append(out.download(q.size).view(np.uint32))
    np.testing.assert_array_equal(outs[0], outs[1])


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_rows_later_tokens_values_do_not_leak(hip_ctx, monkeypatch, bad):
    """A NaN or an infinity in the value row of one of the chunk's tokens shows in
    that token's output and in later ones, and nowhere before, as with one workgroup
    per token."""
    tokens, start, heads, kv_heads = 21, 8190, 8, 2
    cap = start + tokens
    print(f"rows {bad} in a later value row", flush=True)
    q, k, v = inputs(7, tokens, start, cap, heads, kv_heads)
    vf = v.view(np.float16).reshape(cap, kv_heads, D)
    vf[start + 6, 0, 17] = bad
    vf[start + 18, 1, 255] = bad
    ops = kh.NumpyOps(hip_ctx)
    args = (q, k, vf.reshape(-1).view(np.uint16), 0, start, tokens, cap, heads, kv_heads, D)
    got = ops.attention_batched(*args).reshape(tokens, heads, D)
    monkeypatch.setenv("KRAKEN_DECODE_KERNEL", "short")
    one = ops.attention_batched(*args).reshape(tokens, heads, D)
    assert np.isfinite(got[:6]).all() and np.isfinite(got[6:18, 4:]).all()
    assert not np.isfinite(got[6:, :4, 17]).any() and not np.isfinite(got[18:, 4:, 255]).any()
    finite = np.isfinite(one)
    np.testing.assert_array_equal(np.isfinite(got), finite)
    np.testing.assert_allclose(got[finite], one[finite], rtol=0, atol=8e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,start,heads,kv_heads", [
    (40, 3000, 32, 8),   # the several-token kernel's splits, where one token's are one
    (5, 9000, 8, 2),
    (1, 4096, 8, 2),     # one token, split keys
])
@pytest.mark.parametrize("shift", [0, 1, 4])
def test_f16_query_at_any_alignment(hip_ctx, tokens, start, heads, kv_heads, shift):
    """An f16 query is widened into the workspace before these kernels read it, so
    its own alignment changes nothing: the f32 entry's bits."""
    torch = pytest.importorskip("torch")
    print(f"rows f16 query tokens={tokens} heads={heads}/{kv_heads} shift={shift}", flush=True)
    cap = start + tokens
    q, k, v = inputs(11, tokens, start, cap, heads, kv_heads)
    q = q.astype(np.float16)
    want = kh.NumpyOps(hip_ctx).attention_batched(q.astype(np.float32), k, v, 0, start, tokens,
                                                  cap, heads, kv_heads, D)
    held = torch.zeros(q.size + 8, dtype=torch.float16, device="cuda")
    view = held[shift:shift + q.size]
    view.copy_(torch.from_numpy(q))
    torch.cuda.synchronize()
    kb, vb = hip_ctx.buffer(k), hip_ctx.buffer(v)
    out = hip_ctx.buffer(byte_size=4 * q.size)
    hip_ctx.attention_f16q_batched_f16_kv(view, kb, vb, 0, start, tokens, cap, heads, kv_heads, D,
                                          out)
    np.testing.assert_array_equal(out.download(q.size).view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("check", ["test_m0_has_no_other_user",
                                   "test_no_scc_value_lives_across_the_m0_add",
                                   "test_m0_write_never_directly_precedes_an_lds_dma_load"])
def test_rows_copies_own_m0(tmp_path, monkeypatch, check):
    isa = importlib.import_module("test_isa_m0")
    monkeypatch.setitem(isa.EXTRA, "attention_rows.hip", ["-mllvm", "-amdgpu-mfma-vgpr-form"])
    getattr(isa, check)(tmp_path, "attention_rows.hip")
