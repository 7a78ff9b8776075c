"""Rows of a small vocabulary (one launch, the row sorted in registers) against
the oracle: ids and processed distributions around the kernel's sizes, with
ties across every cut (needs an MI355X)."""

from __future__ import annotations

import numpy as np
import pytest

import oracle
from pagellm_amd import _native
from pagellm_amd.params import SamplingParams
from pagellm_amd.sampling import _pack_histories, _pack_params, sample_batch
from parity import compare_rows

pytestmark = pytest.mark.gpu

PARAMS = [
    SamplingParams(temperature=0.0),
    SamplingParams(temperature=0.0, repetition_penalty=1.3),
    SamplingParams(temperature=0.8),
    SamplingParams(top_k=1),
    SamplingParams(top_k=63),
    SamplingParams(temperature=1.7, top_k=2000),
    SamplingParams(top_p=0.9),
    SamplingParams(temperature=0.6, top_p=1e-9),
    SamplingParams(top_p=0.999999, repetition_penalty=1.2),
    SamplingParams(temperature=0.6, top_k=40, top_p=0.95, repetition_penalty=1.1),
    SamplingParams(temperature=3.0, top_k=5, top_p=0.5, repetition_penalty=0.7),
]


def _rows(g, V, dtype):
    """Three shapes per parameter set: smooth, values quantised to half units
    (ties across every cut), a third of the row masked."""
    x = g.normal(0.0, 3.0, (3, len(PARAMS), V))
    x[1] = np.round(2 * x[1]) / 2
    x[2][g.random((len(PARAMS), V)) < 1 / 3] = -np.inf
    x[2][:, V // 2] = 1.0
    params = PARAMS * 3
    hist = [g.integers(0, V, n) for n in g.integers(1, 2100, len(params))]
    return x.reshape(-1, V).astype(dtype), params, hist, g.random(len(params))


# one token; a wave's 64 lanes; one and two tokens a thread; past the last size
@pytest.mark.parametrize("V", [1, 2, 63, 64, 65, 511, 512, 513, 1023, 1024, 1025])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_small_rows(V, dtype):
    g = np.random.default_rng(V)
    x, params, hist, u = _rows(g, V, dtype)
    u[::7] = 0.0
    u[3::7] = 1 - 2.0 ** -53
    print(f"[small] V={V} {np.dtype(dtype).name}", flush=True)
    ids = sample_batch(x, params, uniforms=u, contexts=hist)
    w = dict(logits=x, params=params, contexts=hist, uniforms=u)
    mism, _ = compare_rows(w, range(len(params)), ids, f"small V={V}")
    assert mism == 0

    # the exported distributions, through rows of a wider buffer
    c = _native.default_context()
    c.set_stream(None)
    B = len(params)
    t, k, p, r = _pack_params(params)
    hi, ho = _pack_histories(hist, params, B, V)
    buf = np.full((B, V + 3), np.nan, dtype)
    buf[:, :V] = x
    d = {n: c.to_device(a) for n, a in dict(x=buf, t=t, k=k, p=p, r=r, u=u, hi=hi, ho=ho).items()}
    out, pr = c.empty((B,), np.int32), c.empty((B, V), np.float64)
    c.sample(d["x"].ptr, _native.dtype_code(buf.dtype), V + 3, B, V, d["hi"].ptr, d["ho"].ptr, d["t"].ptr, d["k"].ptr,
             d["p"].ptr, d["r"].ptr, d["u"].ptr, out.ptr, pr.ptr, 0)
    got = pr.download()
    for b in range(B):
        ref = oracle.probs(x[b], params[b], hist[b])
        assert np.array_equal(got[b] > 0, ref > 0), (b, params[b])
        np.testing.assert_allclose(got[b], ref, rtol=1e-13, atol=1e-300)
    nongreedy = [b for b in range(B) if not params[b].greedy]
    assert np.array_equal(out.download()[nongreedy], ids[nongreedy])
