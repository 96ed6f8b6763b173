"""K-quant products of more than 8 tokens with the weights decoded in registers
(kraken-infer_amd/csrc/kquant_mm.hip) at the edges of its tiles and of the rule
that chooses them, against the two-pass form (KRAKEN_KQUANT_GEMM=unfused), whose
fp16 weights come from the exact dequantization that other tests pin.

Both multiply the same fp16 operands.  The tiles that walk K in one chain (128
and 256 rows, and Q6_K's 64) run the same MFMAs in the same order as a two-pass
product without K splits: bit-identical.  The tiles whose four waves split K add
the same products in another order: within TOL * sum |w x|, the bound that
test_gpu_kquant.py derives for either order against the exact product."""
import numpy as np
import pytest

import kquant_cases as kc
import kraken_hip as kh
from test_gpu_kquant import FORMATS, TOL, check_projection, oracle_projection


@pytest.fixture(scope="module")
def ops(hip_ctx):
    return kh.NumpyOps(hip_ctx)


def operands(fmt, rows, cols, tokens):
    w = kc.random_weight_fast(fmt, rows, cols, seed=rows * 3 + cols)
    x = np.random.default_rng(tokens).standard_normal(tokens * cols).astype(np.float32)
    return w, x


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("rows,cols,tokens", [
    (1, 256, 9),        # one row, one K block: three of the four waves have none
    (31, 512, 31), (32, 768, 32), (33, 1280, 33),   # 32 x 32 tiles and their remainders
    (256, 3584, 255),   # the most 32 x 32 tiles with K blocks split 4, 4, 3, 3
    (2049, 256, 127),   # 32 x 64
    (4096, 512, 129),   # 64 x 64
])
def test_split_tiles_against_two_pass(ops, monkeypatch, fmt, rows, cols, tokens):
    print(f"mm split {fmt} {rows}x{cols} tokens={tokens}", flush=True)
    w, x = operands(fmt, rows, cols, tokens)
    got = ops.kquant_matmul(fmt, w, rows, cols, x, tokens)
    if rows * cols * tokens < 2**28:
        want, scale = oracle_projection(fmt, w, rows, cols, x, tokens)
        check_projection(got, want, scale, f"{fmt} {rows}x{cols} T={tokens}")
    monkeypatch.setenv("KRAKEN_KQUANT_GEMM", "unfused")
    two_pass = ops.kquant_matmul(fmt, w, rows, cols, x, tokens).astype(np.float64)
    # |x| <= 6 and sum |w x| >= |w . x|: a floor for the scale of each output.
    scale = np.abs(two_pass).mean() * np.sqrt(cols)
    assert np.abs(got - two_pass).max() <= 2 * TOL * scale


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("rows,cols,tokens", [
    (3585, 1024, 777),   # 128-row tiles, one row and nine tokens past them
    (6100, 512, 900),    # 256-row tiles, partial
    (4100, 256, 640),    # one K block: fewer stages than the pipeline holds
    (4100, 256, 900),    # the same in 256-row tiles (Q4_K, Q5_K)
])
def test_chain_tiles_equal_two_pass(ops, monkeypatch, fmt, rows, cols, tokens):
    print(f"mm chain {fmt} {rows}x{cols} tokens={tokens}", flush=True)
    w, x = operands(fmt, rows, cols, tokens)
    got = ops.kquant_matmul(fmt, w, rows, cols, x, tokens)
    monkeypatch.setenv("KRAKEN_KQUANT_GEMM", "unfused")
    two_pass = ops.kquant_matmul(fmt, w, rows, cols, x, tokens)
    np.testing.assert_array_equal(got.view(np.uint32), two_pass.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,tokens", [
    (4090, 1280, 500),                      # 64-row tiles
    (6100, 512, 257), (12290, 256, 130),    # 128
    (12290, 256, 257), (16390, 512, 200),   # 256
])
def test_q6_chain_tiles_equal_two_pass(ops, monkeypatch, rows, cols, tokens):
    """The shapes for which Q6_K takes them: elsewhere its many-token products stay
    with the two-pass form (mm_us in kquant_mm.hip)."""
    print(f"mm chain q6_k {rows}x{cols} tokens={tokens}", flush=True)
    w, x = operands("q6_k", rows, cols, tokens)
    got = ops.kquant_matmul("q6_k", w, rows, cols, x, tokens)
    monkeypatch.setenv("KRAKEN_KQUANT_GEMM", "unfused")
    two_pass = ops.kquant_matmul("q6_k", w, rows, cols, x, tokens)
    np.testing.assert_array_equal(got.view(np.uint32), two_pass.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,rows,cols,tokens", [
    ("q4_k", 8192, 256, 512), ("q4_k", 8192, 256, 513),      # B tile; 256-row tiles
    ("q5_k", 1024, 3584, 512), ("q5_k", 1024, 3584, 513),    # 32 x 64; two passes, K split
    ("q6_k", 6144, 1024, 567), ("q6_k", 6144, 1024, 568),    # 128 rows; two passes
])
def test_either_side_of_the_estimates(ops, monkeypatch, fmt, rows, cols, tokens):
    """Shapes next to each other that the estimated times send to different forms."""
    print(f"mm estimates {fmt} {rows}x{cols} tokens={tokens}", flush=True)
    w, x = operands(fmt, rows, cols, tokens)
    got = ops.kquant_matmul(fmt, w, rows, cols, x, tokens)
    monkeypatch.setenv("KRAKEN_KQUANT_GEMM", "unfused")
    two_pass = ops.kquant_matmul(fmt, w, rows, cols, x, tokens)
    scale = np.abs(two_pass).mean() * np.sqrt(cols)
    assert np.abs(got - two_pass).max() <= 2 * TOL * scale


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", FORMATS)
def test_group_equals_single(hip_ctx, ops, fmt):
    """Matrices of one format share a launch; a matrix as large as the group's
    largest takes the same tiles on its own."""
    cols, tokens, rows = 1024, 100, [700, 1, 700, 33]
    print(f"mm group {fmt}", flush=True)
    ggml = {"q4_k": 12, "q5_k": 13, "q6_k": 14}[fmt]
    ws = [operands(fmt, r, cols, tokens + i)[0] for i, r in enumerate(rows)]
    x = operands(fmt, 1, cols, tokens)[1]
    outs = [hip_ctx.buffer(byte_size=4 * tokens * r) for r in rows]
    hip_ctx.kquant_matmul_multi([ggml] * 4, [hip_ctx.buffer(w) for w in ws], rows, cols, tokens,
                                hip_ctx.buffer(x), outs)
    for r, w, out in zip(rows, ws, outs):
        got = out.download(tokens * r)
        if r == 700:
            np.testing.assert_array_equal(got, ops.kquant_matmul(fmt, w, r, cols, x, tokens))
        want, scale = oracle_projection(fmt, w, r, cols, x, tokens)
        check_projection(got, want, scale, f"{fmt} group {r} rows")


@pytest.mark.gpu
def test_capture_without_a_grown_workspace():
    """A product that is captured before its context's workspace holds the packed
    inputs: the workspace grows, and replays have the eager result's bits."""
    import torch

    cols, rows, tokens = 1024, 2048, 1024
    w, x = operands("q4_k", rows, cols, tokens)
    wt = torch.from_numpy(np.frombuffer(w.tobytes(), np.uint8).copy()).cuda()
    xt = torch.from_numpy(x).cuda()
    out = torch.empty(tokens * rows, device="cuda")
    ctx = kh.Context()
    stream = torch.cuda.Stream()
    ctx.set_stream(stream.cuda_stream)
    ctx.begin_graph()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        ctx.matmul_q4_k_f32_device(wt, rows, cols, tokens, xt, out)
    got = []
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got.append(out.clone())
    with torch.cuda.stream(stream):
        ctx.matmul_q4_k_f32_device(wt, rows, cols, tokens, xt, out)
    torch.cuda.synchronize()
    for g in got:
        assert torch.equal(g, out)
    del graph
    ctx.commit_graph()
    ctx.close()
