"""The LDS-staged gated delta net recurrence (kraken-infer_amd/csrc/gdn.hip) where it
takes tokens four at a time: every remainder of a group, of the 64 tokens in LDS and
of the rule that hands longer chunks to the chunked kernels; more heads than fit the
GPU at once; non-finite inputs.

Against the oracle within 1e-5: outputs and state are below 2 in size here and each
is a chain of at most `tokens` f32 roundings of 2^-24 of that; a token out of place
misses by 1e-1."""
import numpy as np
import pytest

import kraken_hip as kh
import oracle
from test_gpu_gdn import gdn_inputs


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,hk,hv", [
    (2, 16, 16), (3, 16, 16), (4, 2, 2), (5, 1, 3), (7, 16, 32), (63, 16, 16), (64, 16, 32),
    (66, 16, 16), (127, 4, 4), (160, 16, 32), (161, 16, 32), (96, 16, 48), (97, 16, 48),
    (64, 5, 65),
])
def test_short_chunks_against_oracle(hip_ctx, tokens, hk, hv):
    print(f"gdn short tokens={tokens} heads={hk}/{hv}", flush=True)
    args = gdn_inputs(tokens, tokens, hk, hv, 128, state_scale=0.1)
    out, state = kh.NumpyOps(hip_ctx).gated_delta_net(*args, tokens, hk, hv, 128)
    want, want_state = oracle.gated_delta_net(*args, tokens, hk, hv, 128)
    np.testing.assert_allclose(out, want, rtol=0, atol=1e-5)
    np.testing.assert_allclose(state, want_state, rtol=0, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,hk,hv", [
    (64, 16, 16), (100, 16, 16), (160, 16, 16),
    (64, 2, 4), (130, 2, 6),   # grouped heads, a partial last chunk
])
def test_chunked_kernels_below_their_rule(hip_ctx, monkeypatch, tokens, hk, hv):
    print(f"gdn chunked tokens={tokens} heads={hk}/{hv}", flush=True)
    args = gdn_inputs(tokens, tokens, hk, hv, 128, state_scale=0.1)
    monkeypatch.setenv("KRAKEN_GDN_PREFILL", "chunked")
    out, state = kh.NumpyOps(hip_ctx).gated_delta_net(*args, tokens, hk, hv, 128)
    want, want_state = oracle.gated_delta_net(*args, tokens, hk, hv, 128)
    np.testing.assert_allclose(out, want, rtol=0, atol=1e-4)
    np.testing.assert_allclose(state, want_state, rtol=0, atol=1e-4)


@pytest.mark.gpu
def test_a_tokens_non_finite_query_stays_its_own(hip_ctx):
    tokens, h = 11, 2
    print("gdn NaN and infinity in a query", flush=True)
    q, k, v, g, b, s = gdn_inputs(3, tokens, h, h, 128, state_scale=0.1)
    clean, state = kh.NumpyOps(hip_ctx).gated_delta_net(q, k, v, g, b, s, tokens, h, h, 128)
    q = q.copy()
    q.reshape(tokens, h, 128)[5, 0, 77] = np.nan
    q.reshape(tokens, h, 128)[9, 1, 3] = np.inf
    out, state2 = kh.NumpyOps(hip_ctx).gated_delta_net(q, k, v, g, b, s, tokens, h, h, 128)
    out, clean = out.reshape(tokens, h, 128), clean.reshape(tokens, h, 128)
    hit = np.zeros((tokens, h), bool)
    hit[5, 0] = hit[9, 1] = True
    assert not np.isfinite(out[hit]).any()
    np.testing.assert_array_equal(out[~hit], clean[~hit])
    np.testing.assert_array_equal(state2, state)
