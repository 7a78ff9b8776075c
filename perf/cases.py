"""The calls a user of this framework makes, at the sizes they make them.

Each case is one pass through a public entry point on device-resident data
(the C ABI through ``Context``, or the Python API where the name says so):

  sample   one sampling step of a batch: logits in HBM, packed parameters
           and histories, token ids out
  step     the same step through ``sample_batch``: parameters, uniforms and
           token histories packed on the host, ids back on the host
  probs    the processed distributions of a batch (a speculative round's
           target or draft rows)
  draw     inverse-CDF draws from given distributions
  verify   the accept/resample step of speculative decoding
  head     the final RMSNorm and lm_head product that makes the logits
"""

from __future__ import annotations

import math

import numpy as np
import torch

from pagellm_amd import _native
from pagellm_amd.head import LogitsHead
from pagellm_amd.params import SamplingParams
from pagellm_amd.sampling import abi_params, sample_batch

# Parameters of a batch's rows, by mode.  "mixed": four equal groups of
# requests; "chat": every request the same chat settings; "char": a quarter
# greedy, the rest top-k and top-p; "nucleus": a top_p that keeps most of the
# vocabulary; "spec": a speculative round's sequences, one setting each in turn.
_MIXED = (
    SamplingParams(temperature=0.0),
    SamplingParams(top_k=50),
    SamplingParams(top_p=0.9),
    SamplingParams(temperature=0.6, top_k=40, top_p=0.95, repetition_penalty=1.1),
)
_SPEC = (
    SamplingParams(temperature=0.0),
    SamplingParams(temperature=1.0),
    SamplingParams(temperature=0.8, top_k=30),
    SamplingParams(temperature=1.0, top_p=0.9, repetition_penalty=1.2),
    SamplingParams(temperature=0.7, top_k=50, top_p=0.95, repetition_penalty=1.1),
)
_CHAT = SamplingParams(temperature=0.7, top_k=0, top_p=0.95, repetition_penalty=1.2)
_CHAR = SamplingParams(temperature=0.8, top_k=10, top_p=0.9, repetition_penalty=1.1)
_NUCLEUS = SamplingParams(temperature=1.0, top_k=0, top_p=0.99, repetition_penalty=1.05)


def _row_params(mode: str, rows: int) -> list[SamplingParams]:
    if mode == "mixed":
        return [_MIXED[4 * b // rows] for b in range(rows)]
    if mode == "spec":
        return [_SPEC[b % 5] for b in range(rows)]
    if mode == "char":
        return [_MIXED[0] if 4 * b < rows else _CHAR for b in range(rows)]
    return [_CHAT if mode == "chat" else _NUCLEUS] * rows


def listed() -> list[dict]:
    return [
        # a character-level model's step: the smallest call, launches and latency
        dict(name="sample_char", kind="sample", rows=16, vocab=65, dtype="float32", mode="char", hist=64),
        # a serving step of a 32k-token model, Zipf-shaped rows with chat settings
        dict(name="sample_chat32k", kind="sample", rows=64, vocab=32000, dtype="float32", mode="chat", hist=512),
        # the headline batch: 256 requests of four kinds over a 128k vocabulary
        dict(name="sample_mixed128k", kind="sample", rows=256, vocab=128256, dtype="float32", mode="mixed", hist=2048),
        # the largest batch: nearly the whole of a 152k vocabulary stays in the nucleus
        dict(name="sample_nucleus152k", kind="sample", rows=1024, vocab=152064, dtype="float32", mode="nucleus",
             hist=4096),
        # float64 logits of an odd vocabulary, rows that do not start on 16 bytes
        dict(name="sample_f64_50k", kind="sample", rows=32, vocab=50257, dtype="float64", mode="mixed", hist=300),
        # one engine step with the host in the loop
        dict(name="step_50k", kind="step", rows=48, vocab=50257, dtype="float32", mode="mixed", hist=300),
        # the target rows of a speculative round: 64 sequences, 4 drafts each
        dict(name="probs_round32k", kind="probs", rows=320, vocab=32000, dtype="float32", mode="spec", hist=256),
        # one draft position's draws
        dict(name="draw_32k", kind="draw", rows=64, vocab=32000, dtype="float64"),
        # accept and resample of that round
        dict(name="verify_32k", kind="verify", rows=64, vocab=32000, dtype="float64", k=4),
        # the logits of a full batch
        dict(name="head_256", kind="head", rows=256, vocab=128256, width=4096),
        # the logits of a few interactive requests
        dict(name="head_8", kind="head", rows=8, vocab=128256, width=4096),
        # an odd vocabulary (unaligned weight rows) and a batch between the two
        dict(name="head_odd50k", kind="head", rows=45, vocab=50257, width=1000),
    ]


_MOST_ELEMENTS = 1024 * 152064


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(["sample", "sample", "sample", "step", "probs", "draw", "verify", "head", "head"])
    if kind == "head":
        c = dict(kind=kind, rows=_log_int(rng, 1, 256), vocab=_log_int(rng, 65, 128256), width=_log_int(rng, 64, 4096))
        if rng.random() < 0.5:  # sizes as models have them, in whole tiles
            c["vocab"], c["width"] = -(-c["vocab"] // 128) * 128, -(-c["width"] // 64) * 64
            c["vocab"] = min(c["vocab"], 128256)
        return c
    c = dict(kind=kind, rows=_log_int(rng, 1, 1024 if kind == "sample" else 320), vocab=_log_int(rng, 65, 152064))
    c["rows"] = max(1, min(c["rows"], _MOST_ELEMENTS // (4 * c["vocab"]) if kind != "sample" else c["rows"]))
    if kind == "verify":
        c["k"] = rng.randint(0, 8)
        c["rows"] = max(1, min(c["rows"], 64))
        c["dtype"] = rng.choice(["float64", "float64", "float32"])
        return c
    if kind == "draw":
        c["dtype"] = rng.choice(["float64", "float64", "float32"])
        return c
    c["dtype"] = rng.choice(["float32", "float32", "float32", "float64"])
    c["mode"] = "spec" if kind == "probs" else rng.choice(["mixed", "mixed", "chat", "char", "nucleus"])
    c["hist"] = _log_int(rng, 1, 4096)
    if kind != "sample":
        c["hist"] = min(c["hist"], 512)
    if c["dtype"] == "float64":  # twice the bytes
        c["rows"] = max(1, c["rows"] // 2)
    return c


# ------------------------------------------------------------------- inputs


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) % (1 << 62))
    return g


def _zipf(g, rows: int, V: int, s: float, noise: float):
    """Logits -s ln(rank) + N(0, noise^2), the ranks in random order per row,
    and each row's token of rank r."""
    order = torch.rand((rows, V), generator=g, device="cuda").argsort(dim=1)
    y = -s * torch.log(torch.arange(1, V + 1, device="cuda", dtype=torch.float32)).expand(rows, V)
    x = torch.empty((rows, V), device="cuda").scatter_(1, order, y)
    x += noise * torch.randn((rows, V), generator=g, device="cuda")
    return x, order


def _logits(case: dict, seed: int):
    """(logits [rows, V], histories int64 [rows, hist]) of the case's mode."""
    g = _gen(seed)
    B, V, H, mode = case["rows"], case["vocab"], case["hist"], case["mode"]
    if mode in ("chat", "nucleus"):
        s, noise = (1.1, 0.5) if mode == "chat" else (1.0, 0.3)
        x, order = _zipf(g, B, V, s, noise)
        cdf = torch.arange(1, V + 1, device="cuda", dtype=torch.float64).pow(-s).cumsum(0)
        u = torch.rand((B, H), generator=g, device="cuda", dtype=torch.float64) * cdf[-1]
        hist = order.gather(1, torch.searchsorted(cdf, u).clamp_(max=V - 1))
    else:
        x = (3.0 if mode == "mixed" else 2.0) * torch.randn((B, V), generator=g, device="cuda")
        if mode == "mixed":  # a few likely tokens
            n = min(8, V)
            top = torch.rand((B, V), generator=g, device="cuda").topk(n, dim=1).indices
            x.scatter_add_(1, top, torch.full((B, n), 10.0, device="cuda"))
        hist = torch.randint(0, V, (B, H), generator=g, device="cuda")
    u = torch.rand(B, generator=g, device="cuda", dtype=torch.float64)
    if case["dtype"] == "float64":  # float64 logits use all of their bits
        x = x.double() + 1e-9 * torch.randn((B, V), generator=g, device="cuda", dtype=torch.float64)
    return x, hist, u


def _softmax_rows(g, shape, scale: float, dtype):
    return torch.softmax(scale * torch.randn(shape, generator=g, device="cuda", dtype=torch.float64), dim=-1).to(dtype)


def _verify_inputs(case: dict, seed: int):
    g = _gen(seed)
    B, k, V = case["rows"], case["k"], case["vocab"]
    target = 2.0 * torch.randn((B, k + 1, V), generator=g, device="cuda", dtype=torch.float64)
    q = target[:, :k] + 0.5 * torch.randn((B, k, V), generator=g, device="cuda", dtype=torch.float64)
    p, q = torch.softmax(target, dim=-1), torch.softmax(q, dim=-1)
    c = q.cumsum(-1)
    u = torch.rand((B, k, 1), generator=g, device="cuda", dtype=torch.float64)
    draft = torch.searchsorted(c, u * c[..., -1:], right=True).clamp_(max=V - 1)[..., 0]
    accept = torch.rand((B, k), generator=g, device="cuda", dtype=torch.float64)
    w = torch.rand(B, generator=g, device="cuda", dtype=torch.float64)
    dt = getattr(torch, case["dtype"])
    return p.to(dt), q.to(dt), draft.to(torch.int32), accept, w


def _head_inputs(case: dict, seed: int):
    g = _gen(seed)
    N, D, V = case["rows"], case["width"], case["vocab"]
    h = torch.randn((N, D), generator=g, device="cuda")
    norm = 1 + 0.1 * torch.randn(D, generator=g, device="cuda")
    W = torch.randn((D, V), generator=g, device="cuda").mul_(0.02)
    return h, norm, W


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    s = dict(kind=kind, case=case, ctx=_native.default_context())
    if kind == "head":
        h, norm, W = _head_inputs(case, seed)
        s.update(h=h, head=LogitsHead(norm, W, 1e-5), out=torch.empty((case["rows"], case["vocab"]), device="cuda"))
        return s
    B, V = case["rows"], case["vocab"]
    s["ids"] = torch.empty(B, dtype=torch.int32, device="cuda")
    if kind == "verify":
        p, q, draft, accept, w = _verify_inputs(case, seed)
        s.update(p=p, q=q, draft=draft, accept=accept, w=w,
                 toks=torch.empty((B, case["k"] + 1), dtype=torch.int32, device="cuda"))
        return s
    if kind == "draw":
        g = _gen(seed)
        s.update(p=_softmax_rows(g, (B, V), 2.0, getattr(torch, case["dtype"])),
                 u=torch.rand(B, generator=g, device="cuda", dtype=torch.float64))
        return s
    x, hist, u = _logits(case, seed)
    params = _row_params(case["mode"], B)
    s["x"] = x
    if kind == "step":
        s.update(params=params, contexts=[row.tolist() for row in hist.cpu().numpy()], u=u.cpu().numpy())
        return s
    a = abi_params(params)
    s.update({name: torch.from_numpy(v).cuda() for name, v in a.items()})
    # the histories of the rows whose penalty is active
    on = a["repetition_penalty"] != 1.0
    off = np.concatenate([[0], np.cumsum(np.where(on, case["hist"], 0))]).astype(np.int64)
    s["hist_off"] = torch.from_numpy(off).cuda()
    s["hist_ids"] = hist[torch.from_numpy(on).cuda()].to(torch.int32).reshape(-1).contiguous()
    s["u"] = u
    nuc = (a["temperature"] != 0) & ((a["top_k"] == 0) | (a["top_k"] >= V)) & (a["top_p"] >= 0.98) & (a["top_p"] < 1)
    s["flags"] = 0
    if kind == "sample" and nuc.any():
        s["flags"] = _native.PLH_SAMPLE_NUCLEUS | (_native.PLH_SAMPLE_NUCLEUS_ONLY if nuc.all() else 0)
    s["probs"] = torch.empty((B, V), dtype=torch.float64, device="cuda") if kind == "probs" else None
    return s


def run(s: dict):
    kind, case, c = s["kind"], s["case"], s["ctx"]
    if kind == "head":
        return s["head"](s["h"], out=s["out"])
    if kind == "step":
        return sample_batch(s["x"], s["params"], contexts=s["contexts"], uniforms=s["u"])
    c.set_stream(torch.cuda.current_stream().cuda_stream)
    B, V, code = case["rows"], case["vocab"], _native.dtype_code(np.dtype(case["dtype"]))
    if kind == "verify":
        k = case["k"]
        c.verify(s["p"].data_ptr(), s["q"].data_ptr() if k else None, code, B, k, V,
                 s["draft"].data_ptr() if k else None, s["accept"].data_ptr() if k else None, s["w"].data_ptr(), False,
                 s["toks"].data_ptr(), s["ids"].data_ptr())
        return s["toks"], s["ids"]
    if kind == "draw":
        c.draw(s["p"].data_ptr(), code, V, B, V, s["u"].data_ptr(), s["ids"].data_ptr())
        return s["ids"]
    c.sample(s["x"].data_ptr(), code, V, B, V, s["hist_ids"].data_ptr() if s["hist_ids"].numel() else None,
             s["hist_off"].data_ptr() if s["hist_ids"].numel() else None, s["temperature"].data_ptr(),
             s["top_k"].data_ptr(), s["top_p"].data_ptr(), s["repetition_penalty"].data_ptr(), s["u"].data_ptr(),
             s["ids"].data_ptr(), s["probs"].data_ptr() if kind == "probs" else None, s["flags"])
    return (s["ids"], s["probs"]) if kind == "probs" else s["ids"]


def work(case: dict) -> dict:
    kind, B, V = case["kind"], case["rows"], case["vocab"]
    if kind == "head":
        D = case["width"]
        return {"bytes": 4 * (D * V + B * D + D + B * V), "flops": 2 * B * D * V}
    e = 8 if case["dtype"] == "float64" else 4
    if kind == "verify":
        # the distributions at the position where the row stops, and the tests' gathers
        return {"bytes": B * (2 * e * V + (2 * e + 12) * case["k"] + 16), "flops": 3 * B * V}
    if kind == "draw":
        return {"bytes": B * (e * V + 12), "flops": B * V}
    on = sum(p.repetition_penalty != 1.0 for p in _row_params(case["mode"], B))
    out = 8 * B * V if kind == "probs" else 0
    return {"bytes": e * B * V + out + 4 * case["hist"] * on + 48 * B, "flops": 4 * B * V}


def tolerance(case: dict):
    if case["kind"] == "head":
        # float32 products summed in float32, in any order
        return {"rel": 4e-6, "max": 4e-5}
    if case["kind"] == "probs":
        # float64 throughout: the rounding of z / T, of an exp and of the normaliser's sum
        return {"rel": 2e-15, "max": 4e-14}
    return "exact"


# ------------------------------------------------- the same in plain float64


def _exact_probs(x, p: SamplingParams, hist):
    z = x.double().clone()
    V = z.numel()
    if p.repetition_penalty != 1.0 and hist.numel():
        ids = hist.unique()
        v = x[ids].double()
        z[ids] = torch.where(v > 0, v / p.repetition_penalty, v * p.repetition_penalty)
    if p.temperature == 0:
        out = torch.zeros_like(z)
        out[(z == z.max()).nonzero()[0, 0]] = 1.0
        return out
    z = z / p.temperature
    if 0 < p.top_k < V:
        z = torch.where(z >= z.topk(p.top_k).values[-1], z, -math.inf)
    e = torch.exp(z - z.max())
    e = e / e.sum()
    if p.top_p < 1.0:
        v, order = e.sort(descending=True, stable=True)
        keep = v.cumsum(0) - v < p.top_p
        keep[0] = True
        e = torch.zeros_like(e).scatter_(0, order[keep], v[keep])
        e = e / e.sum()
    return e


def exact(case: dict, seed: int):
    """What run() returns, in plain float64 (None for token ids)."""
    if case["kind"] == "head":
        h, norm, W = _head_inputs(case, seed)
        h = h.double()
        a = h / torch.sqrt((h * h).mean(dim=1, keepdim=True) + 1e-5) * norm.double()
        return torch.cat([a @ W[:, v:v + 16384].double() for v in range(0, case["vocab"], 16384)], dim=1)
    if case["kind"] == "probs":
        x, hist, _ = _logits(case, seed)
        params = _row_params(case["mode"], case["rows"])
        return None, torch.stack([_exact_probs(x[b], params[b], hist[b]) for b in range(case["rows"])])
    return None
