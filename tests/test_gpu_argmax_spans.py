"""argmax_prob at the edges of its first phase (kraken-infer_amd/csrc/kquant.hip): 1024
values per workgroup up to 256 workgroups, 4096 above.  The index exactly, the
probability within 1e-5 as test_gpu_kquant.py holds it (an f32 sum of exponentials)."""
import numpy as np
import pytest

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
