"""argmax_prob at the edges of its first phase (kraken-infer_amd/csrc/kquant.hip): 1024
values per workgroup up to 256 workgroups, 4096 above.  The index exactly, the
probability within 1e-5 as test_gpu_kquant.py holds it (an f32 sum of exponentials)."""
import numpy as np
import pytest

import kquant_cases as kc
import kraken_hip as kh
import oracle


@pytest.mark.gpu
@pytest.mark.parametrize("size", [17408, 17409, 262143, 262144, 262145, 1048577])
def test_argmax_span_edges(hip_ctx, size):
    print(f"argmax size={size}", flush=True)
    ops = kh.NumpyOps(hip_ctx)
    v = np.random.default_rng(size).standard_normal(size).astype(np.float32)
    for at in ([size - 1], [1023, 1024], [0, size - 1], [size - 257, size - 2]):
        w = v.copy()
        w[at] = 9.0
        w[at[0] // 2 + 1] = np.nan if at[0] > 1024 else w[at[0] // 2 + 1]
        assert ops.argmax(w) == oracle.argmax(w) == at[0]
        token, p = ops.argmax(w, probability=True)
        want_token, want = oracle.argmax(w, probability=True)
        assert token == want_token
        if np.isfinite(w).all():
            assert abs(p - want) <= 1e-5 * want
        else:
            assert p == want == 0.0


@pytest.mark.gpu
def test_top1_does_not_depend_on_the_workspace():
    """261700 logits and their candidates fit a workspace of 1 MiB with 4096 values
    per candidate and not with 1024: the same probability, bit for bit, from a new
    context and from one whose workspace has grown."""
    rows, cols = 261700, 256
    print(f"top1 rows={rows} by workspace", flush=True)
    w = kc.random_weight_fast("q4_k", rows, cols, seed=5)
    x = np.random.default_rng(5).standard_normal(cols).astype(np.float32) / 16
    got = []
    for grown in (False, True):
        ctx = kh.Context()
        ops = kh.NumpyOps(ctx)
        if grown:
            ops.kquant_matmul("q5_k", kc.random_weight_fast("q5_k", 64, 1024, 1), 64, 1024,
                              np.ones(2048 * 1024, np.float32), 2048)
        token, p = ops.kquant_top1("q4_k", w, rows, cols, x, probability=True)
        got.append((token, np.float32(p).view(np.uint32)))
        ctx.close()
    assert got[0] == got[1]
