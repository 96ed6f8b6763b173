"""Calls captured into a HIP graph by a context whose workspace does not yet hold
what they need: every replay gives the bits of the eager call, whatever the context
did before (the kernel and the split of its work follow from the arguments alone)."""
import numpy as np
import pytest

import kquant_cases as kc
import kraken_hip as kh

GGML = {"q4_k": 12, "q5_k": 13, "q6_k": 14}


def captured_and_eager(call, out, first=None):
    """`call(ctx)` captured on a fresh context (after the eager call `first`, if any),
    replayed three times with the output cleared before each; then the eager result
    of another context."""
    import torch

    stream = torch.cuda.Stream()
    fresh, other = kh.Context(), kh.Context()
    for ctx in (fresh, other):
        ctx.set_stream(stream.cuda_stream)
    if first is not None:
        first(fresh)
    torch.cuda.synchronize()
    fresh.begin_graph()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        call(fresh)
    fresh.commit_graph()
    replays = []
    for _ in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        replays.append(out.clone())
        call(fresh)  # eager work between the replays
    out.fill_(float("nan"))
    torch.cuda.synchronize()
    call(other)
    eager = out.clone()
    torch.cuda.synchronize()
    del graph
    fresh.close()
    other.close()
    assert torch.isfinite(eager).all()
    for r in replays:
        assert torch.equal(r, eager)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,rows,cols,tokens,up,residual", [
    ("q4_k", 2048, 1024, 1024, False, False),
    ("q4_k", 1024, 2048, 1024, False, False),  # few tiles: the older form splits K
    ("q4_k", 1024, 3584, 48, True, True),
    ("q5_k", 6144, 1024, 171, False, False),
    ("q6_k", 1024, 3584, 48, True, True),
])
def test_captured_products(fmt, rows, cols, tokens, up, residual):
    import torch

    print(f"captured product {fmt} {rows}x{cols} tokens={tokens} up={up}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(rows + tokens)
    w = torch.from_numpy(kc.random_weight_fast(fmt, rows, cols, seed=7)).cuda()
    x, u = (torch.randn(tokens * cols, generator=gen, device="cuda") for _ in range(2))
    r = torch.randn(tokens * rows, generator=gen, device="cuda")
    out = torch.empty(tokens * rows, device="cuda")

    def call(ctx):
        ctx.kquant_matmul_fused_f32(GGML[fmt], w, rows, cols, tokens, x, u if up else None,
                                    r if residual else None, out)

    captured_and_eager(call, out)


@pytest.mark.gpu
def test_captured_group_of_products():
    import torch

    rows, cols, tokens = [2048, 16], 1024, 700
    print("captured group of products", flush=True)
    ws = [torch.from_numpy(kc.random_weight_fast("q4_k", n, cols, seed=n)).cuda() for n in rows]
    x = torch.randn(tokens * cols, device="cuda")
    out = torch.empty(tokens * sum(rows), device="cuda")
    outs = [out[:tokens * rows[0]], out[tokens * rows[0]:]]
    captured_and_eager(
        lambda ctx: ctx.kquant_matmul_multi([12, 12], ws, rows, cols, tokens, x, outs), out)


@pytest.mark.gpu
@pytest.mark.parametrize("grown", [False, True])
@pytest.mark.parametrize("kind", ["f16_cache", "f16_cache_f16_query", "f32_cache"])
def test_captured_attention_over_several_tokens(kind, grown):
    """With no workspace, and with one that holds the query's f32 copy or a few
    splits but not what the call asks for."""
    import torch

    print(f"captured attention {kind} grown={grown}", flush=True)
    f16 = kind != "f32_cache"
    tokens, start, heads, kv_heads, d = (37, 6144, 16, 4, 256) if f16 else (100, 500, 16, 8, 128)
    cap = start + tokens
    gen = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn(tokens * heads * d, generator=gen, device="cuda")
    k, v = (torch.randn(cap * kv_heads * d, generator=gen, device="cuda") for _ in range(2))
    out = torch.empty(tokens * heads * d, device="cuda")
    if f16:
        k, v = k.half(), v.half()
    name = "attention_f32_batched_f16_kv" if f16 else "attention_f32_batched"
    if kind == "f16_cache_f16_query":
        name, q = "attention_f16q_batched_f16_kv", q.half()

    def call(ctx):
        ctx.call(name, q, k, v, 0, start, tokens, cap, heads, kv_heads, d, out)

    def grow(ctx):  # one megabyte
        values = torch.randn(20000, device="cuda")
        torch.cuda.synchronize()
        ctx.argmax_f32_i32(values, 20000, torch.empty(1, dtype=torch.int32, device="cuda"))

    captured_and_eager(call, out, grow if grown else None)
