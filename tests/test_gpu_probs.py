"""The processed distributions of rows past the small vocabularies (one
workgroup per row, the exps kept in the row's output) against the oracle:
distributions and ids around the kernel's block sizes, with ties across every
cut (needs an MI355X)."""

from __future__ import annotations

import numpy as np
import pytest

import oracle
from pagellm_amd import _native
from pagellm_amd.params import SamplingParams
from pagellm_amd.sampling import _pack_histories, _pack_params
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
    """Three shapes per parameter set: smooth, a few dozen values (ties across
    every cut), a third of the row masked."""
    x = g.normal(0.0, 3.0, (3, len(PARAMS), V))
    x[1] = np.round(2 * x[1]) / 2
    x[2][g.random((len(PARAMS), V)) < 1 / 3] = -np.inf
    x[2][:, V // 2] = 1.0
    params = PARAMS * 3
    hist = [g.integers(0, V, n) for n in g.integers(1, 2100, len(params))]
    return x.reshape(-1, V).astype(dtype), params, hist, g.random(len(params))


# first past the small kernel; a block of 1024 threads (float64: 2048 tokens,
# float32: 4096) less one, whole and with one to three tokens past the last
# 16-byte vector; more blocks than are loaded at once; an odd vocabulary
@pytest.mark.parametrize("V", [1025, 2049, 4095, 4096, 4097, 8192, 8194, 16387, 32000, 50257])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_probs_rows(V, dtype):
    g = np.random.default_rng(V)
    x, params, hist, u = _rows(g, V, dtype)
    u[::7] = 0.0
    u[3::7] = 1 - 2.0 ** -53
    if V > 20000:  # the oracle sorts every row
        keep = np.arange(0, len(params), 2)
        x, params, hist, u = x[keep], [params[i] for i in keep], [hist[i] for i in keep], u[keep]
    print(f"[probs] V={V} {np.dtype(dtype).name}", flush=True)
    c = _native.default_context()
    c.set_stream(None)
    B = len(params)
    t, k, p, r = _pack_params(params)
    hi, ho = _pack_histories(hist, params, B, V)
    buf = np.full((B, V + 3), np.nan, dtype)
    buf[:, :V] = x
    d = {n: c.to_device(a) for n, a in dict(x=buf, t=t, k=k, p=p, r=r, u=u, hi=hi, ho=ho).items()}
    out, pr = c.empty((B,), np.int32), c.to_device(np.full(B * V + 4, -7.0))
    c.sample(d["x"].ptr, _native.dtype_code(buf.dtype), V + 3, B, V, d["hi"].ptr, d["ho"].ptr, d["t"].ptr, d["k"].ptr,
             d["p"].ptr, d["r"].ptr, d["u"].ptr, out.ptr, pr.ptr, 0)
    got = pr.download()
    assert np.all(got[B * V:] == -7.0)  # nothing past the last row
    got = got[:B * V].reshape(B, V)
    for b in range(B):
        ref = oracle.probs(x[b], params[b], hist[b])
        assert np.array_equal(got[b] > 0, ref > 0), (b, params[b])
        np.testing.assert_allclose(got[b], ref, rtol=1e-13, atol=1e-300)
    w = dict(logits=x, params=params, contexts=hist, uniforms=u)
    mism, _ = compare_rows(w, [b for b in range(B) if not params[b].greedy], out.download(), f"probs V={V}")
    assert mism == 0
    if V <= 8192:  # ids alone come from the same kernel, with the row in LDS
        ids = c.empty((B,), np.int32)
        c.sample(d["x"].ptr, _native.dtype_code(buf.dtype), V + 3, B, V, d["hi"].ptr, d["ho"].ptr, d["t"].ptr, d["k"].ptr,
                 d["p"].ptr, d["r"].ptr, d["u"].ptr, ids.ptr, None, 0)
        assert np.array_equal(ids.download(), out.download())


@pytest.mark.parametrize("V", [8192, 32000])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_rows_sum_to_one(V, dtype):
    """The rows' exact sums are off by the normaliser's rounding and that of its
    reciprocal (rms over the rows): pairwise sums over waves and lanes stay
    within 1e-16, waves added one after another exceed it."""
    g = np.random.default_rng(V)
    B = 192
    x = (2 * g.standard_normal((B, V))).astype(dtype)
    print(f"[probs] sums V={V} {np.dtype(dtype).name}", flush=True)
    c = _native.default_context()
    c.set_stream(None)
    t, k, p, r = _pack_params([SamplingParams()] * B)
    d = {n: c.to_device(a) for n, a in dict(x=x, t=t, k=k, p=p, r=r, u=np.full(B, 0.5)).items()}
    out, pr = c.empty((B,), np.int32), c.empty((B, V), np.float64)
    c.sample(d["x"].ptr, _native.dtype_code(x.dtype), V, B, V, None, None, d["t"].ptr, d["k"].ptr, d["p"].ptr, d["r"].ptr,
             d["u"].ptr, out.ptr, pr.ptr, 0)
    off = pr.download().astype(np.longdouble).sum(axis=1) - 1
    rms = float(np.sqrt(np.mean(off ** 2)))
    print(f"[probs] rms {rms:.2e}", flush=True)
    assert rms < 1e-16, rms
