"""GPU parity of the logits producer (``plh_rmsnorm_lm_head``) against the
CPU oracle and against torch's float32 product, and the head -> sampler chain
with the logits kept in HBM (needs an MI355X).

Tolerance: float32 products summed in a different order than numpy's BLAS
(or hipBLAS) differ by rounding only, which scales with
``sum_d |a[n, d]| |W[d, v]|`` (``oracle.head_error_bound``); every logit must
be within 1e-5 of that bound (a wrong index or a dropped term is off by
O(1) of it).  The reference's own model tests compare float32 logits at
rtol = atol = 1e-4 (``tests/unit/test_model.py:55``)."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle
from pagellm_amd import _native
from pagellm_amd import head as H

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _case(seed, N, D, V, scale=1.0):
    g = np.random.default_rng(seed)
    h = (scale * g.standard_normal((N, D))).astype(np.float32)
    norm = (1 + 0.1 * g.standard_normal(D)).astype(np.float32)
    W = (0.02 * g.standard_normal((D, V))).astype(np.float32)
    return h, norm, W


@pytest.mark.parametrize("N,D,V", [
    (1, 128, 65),        # the reference model's width, the character vocabulary
    (3, 100, 1000),      # D not a multiple of the 32-wide k stage, ragged V tile
    (300, 64, 513),      # two row tiles, the second ragged
    (256, 128, 4096),    # full row tile, V on the vector-load path
    (17, 4096, 300),     # deep k loop
    (5, 1, 7),           # one column of k
    (4097, 520, 65),     # more rows than are ever summed over slices of k
])
def test_head_matches_oracle(N, D, V):
    print(f"[head] N={N} D={D} V={V}", flush=True)
    h, norm, W = _case(N * 7 + D, N, D, V)
    got = H.rms_norm_lm_head(h, norm, W, 1e-5)
    ref = oracle.lm_head_logits(h, norm, W, 1e-5)
    bound = oracle.head_error_bound(h, norm, W, 1e-5)
    assert got.shape == (N, V) and got.dtype == np.float32
    err = np.abs(got.astype(np.float64) - ref)
    assert np.all(err <= TOL * bound + 1e-30), float(np.max(err / (bound + 1e-30)))
    np.testing.assert_allclose(got, ref, rtol=1e-4, atol=1e-4)


def _plan(N, D, V):
    """(rows per workgroup, slices of k) that the library picks for the device."""
    import torch

    f = ctypes.CDLL(str(_native.LIB_PATH))["_ZN3plh9head_planEiiili"]  # plh::head_plan
    f.restype, f.argtypes = ctypes.c_uint64, [ctypes.c_int] * 3 + [ctypes.c_int64, ctypes.c_int]
    r = f(N, D, V, V, torch.cuda.get_device_properties(0).multi_processor_count)
    return r & 0xffffffff, r >> 32


# (1, 16, 17, 32): the few-rows kernels, in one and several slices of k; 33 on:
# the split kernels, in tiles of 64 rows (and at 70 000 columns of 128), with
# ragged and whole row tiles.  test_tile_plans has the other plans.
@pytest.mark.parametrize("N", [1, 16, 17, 32, 33, 64, 65, 129, 256])
@pytest.mark.parametrize("D,V", [
    (8, 127),     # one column short of a workgroup; k ends in a ragged group (16 rows) or a whole one (32)
    (128, 128),   # one workgroup, whole groups and stages
    (129, 257),   # the last workgroup's columns overlap the one's before; one k past the whole groups
    (1000, 333),  # several slices of k, the last one ragged
    (40, 70000),  # enough columns for one slice at every N
])
def test_row_counts_and_edges(N, D, V):
    """Every kernel on W, h and out rows of odd strides (no 16-byte alignment
    anywhere), nothing written outside out."""
    import torch

    print(f"[head] edges N={N} D={D} V={V}", flush=True)
    h, norm, W = _case(N + D, N, D, V)
    wb = torch.full((D, V + 3), float("nan"), device="cuda")
    wb[:, 1:V + 1] = torch.from_numpy(W).cuda()
    hb = torch.full((N, D + 1), float("nan"), device="cuda")
    hb[:, :D] = torch.from_numpy(h).cuda()
    ob = torch.full((N + 1, V + 5), 7.0, device="cuda")
    H.rms_norm_lm_head(hb[:, :D], torch.from_numpy(norm).cuda(), wb[:, 1:V + 1], 1e-5, out=ob[:N, :V])
    got = ob.cpu().numpy()
    bound = oracle.head_error_bound(h, norm, W, 1e-5)
    err = np.abs(got[:N, :V].astype(np.float64) - oracle.lm_head_logits(h, norm, W, 1e-5))
    assert np.all(err <= TOL * bound + 1e-30), float(np.max(err / (bound + 1e-30)))
    assert np.all(got[N:] == 7.0) and np.all(got[:, V:] == 7.0)


@pytest.mark.parametrize("N", [8, 40])  # the fp32 kernel and the bf16 split
@pytest.mark.parametrize("D,V", [(64, 70000), (512, 300)])  # one slice of k, and several
def test_values_at_the_ends_of_float32(N, D, V):
    """Infinities, NaN, values next to overflow and subnormal-sized results:
    the same kinds of value as float32 products and sums give."""
    h, norm, W = _case(5, N, D, V)
    W[3, 7] = np.inf        # +-inf in column 7
    W[4, 9], W[5, 9] = np.inf, -np.inf   # inf - inf somewhere in column 9
    W[:, 11] = 3.3e38       # overflows on the way for some rows
    W[:, 13] *= np.float32(1e-36)   # tiny: its bf16 parts underflow
    W[:, 14] = 0.0
    h[2, 1] = np.nan        # a whole NaN row
    got = H.rms_norm_lm_head(h, norm, W, 1e-5)
    with np.errstate(all="ignore"):
        a = oracle.rms_norm(h, norm, np.float32(1e-5)).astype(np.float64)
        ref = a @ W.astype(np.float64)
    ok = np.arange(N) != 2
    assert np.isnan(got[2]).all() and np.isfinite(got[ok][:, :7]).all()
    assert np.array_equal(got[ok, 7], np.sign(a[ok, 3]) * np.inf)
    same = np.sign(a[ok, 4]) != np.sign(a[ok, 5])
    assert np.array_equal(got[ok, 9][same], (np.sign(a[ok, 4]) * np.inf)[same]) and np.isnan(got[ok, 9][~same]).all()
    over = np.abs(ref[ok, 11]) > 3.5e38  # float32's largest is 3.40e38; partial sums of the rest may overflow too
    assert not np.isfinite(got[ok, 11][over]).any()
    bound = np.abs(a) @ np.abs(W.astype(np.float64))
    # a product of 1e-38 is rounded to float32's subnormal step, 2^-149
    assert np.all(np.abs(got[ok, 13] - ref[ok, 13]) <= TOL * bound[ok, 13] + D * 2.0 ** -149)
    assert np.all(got[ok, 14] == 0.0)
    rest = np.setdiff1d(np.arange(V), [7, 9, 11, 13, 14])
    err = np.abs(got[ok][:, rest] - ref[ok][:, rest])
    assert np.all(err <= TOL * bound[ok][:, rest] + 1e-30)


@pytest.mark.parametrize("N,D,V", [
    (40, 72, 70001),      # 64-row tile, k and columns ragged
    (40, 1000, 333),      # ... in slices of k
    (100, 1016, 70001),   # 128-row tile
    (200, 1000, 128255),  # 256-row tile
])
def test_nothing_past_the_end_of_lm_head_is_read(N, D, V):
    """What lies behind the matrix in memory (here: rows of the same
    allocation) changes no bit of the logits.  A value read there would meet a
    zero of act, but for NaN and infinities, after which the element is formed
    again in another order."""
    import torch

    print(f"[head] tail N={N} D={D} V={V}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(D)
    buf = torch.randn((D + 48, V), generator=g, device="cuda")
    buf[:D] *= 0.02
    W = buf[:D]
    norm = 1 + 0.1 * torch.randn(D, generator=g, device="cuda")
    h = torch.randn((N, D), generator=g, device="cuda")
    ref = None
    for tail in (0.0, float("nan"), float("inf"), 3e38):
        buf[D:] = tail
        got = H.rms_norm_lm_head(h, norm, W, 1e-5)
        ref = got.clone() if ref is None else ref
        assert torch.equal(got, ref), tail


@pytest.mark.parametrize("N,D,V", [(8, 64, 1000), (40, 64, 70000), (40, 512, 300)])  # few rows; one slice, several
@pytest.mark.parametrize("small", ["weights", "rows", "neither"])
def test_small_operands_against_large_ones(N, D, V, small):
    """Operands whose low bits (or all of them) lie below bf16's range, with
    ordinary logits: the other operand is large; and logits of 2^40.  Limit: a float32 sum in any
    order is within D * 2^-24 of the bound, and each factor of act adds a
    rounding or two (TOL covers both)."""
    print(f"[head] small {small} N={N} D={D} V={V}", flush=True)
    h, norm, W = _case(23, N, D, V)
    if small == "weights":
        norm *= np.float32(2.0 ** 64)
        W = W * np.float32(2.0 ** -60)  # ordinary columns of such a matrix
        for c, t in enumerate((124, 112, 104, 140, 126, 118)):
            W[:, 3 + 40 * c] = (50 * W[:, 3 + 40 * c].astype(np.float64) * 2.0 ** (60 - t)).astype(np.float32)
    elif small == "neither":
        norm *= np.float32(2.0 ** 42)
    else:
        norm *= np.float32(2.0 ** -124)
        W = W * np.float32(2.0 ** 64)
    a = oracle.rms_norm(h, norm, np.float32(1e-5)).astype(np.float64)
    ref, bound = a @ W.astype(np.float64), np.abs(a) @ np.abs(W.astype(np.float64))
    got = H.rms_norm_lm_head(h, norm, W, 1e-5)
    # act is rounded to float32's subnormal step, and so is each product
    step = 2.0 ** -149 * (np.abs(W.astype(np.float64)).sum(0) + D) if small == "rows" else D * 2.0 ** -149
    assert np.all(np.abs(got - ref) <= TOL * bound + step), float(np.max(np.abs(got - ref) / (bound + step)))


@pytest.mark.parametrize("N,D,V", [(40, 1, 4096), (40, 2, 4096), (40, 3, 4096), (40, 4, 4096), (40, 8, 4096),
                                   (40, 64, 60000), (40, 1000, 333), (200, 1000, 50257), (256, 4096, 60000)])
def test_sums_of_like_signs(N, D, V):
    """Sums of D products in U(1, 4), where no error cancels: the 2-norm error
    against float64 is within that of D float32 additions, whose roundings
    (uniform, 2^-24 / sqrt(3) of the running sum) give 2^-24 sqrt(D) / 3, or one
    last bit of the result for short sums."""
    import torch

    print(f"[head] like signs N={N} D={D} V={V}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(D)
    W = 1 + torch.rand((D, V), generator=g, device="cuda")
    a = 1 + torch.rand(D, generator=g, device="cuda")
    got = H.rms_norm_lm_head(torch.ones((N, D), device="cuda"), a, W, 0.0).double()  # r = 1: act is a
    ref = a.double() @ W.double()
    err = float((got - ref).norm() / ref.norm() / N ** 0.5)
    assert err <= 2.0 ** -24 * max(1.0, D ** 0.5 / 3), err * 2 ** 24


@pytest.mark.parametrize("N,V,ldw", [(2_100_000, 3, 3), (2_100_000, 3, (1 << 24) + 4), (70, 200, (1 << 24) + 4)])
def test_many_rows_and_rows_of_lm_head_far_apart(N, V, ldw):
    """The few-rows kernel over many row tiles: short sums, and rows of W that
    lie more than 64 MB apart (r, act and the sums: at most 8 roundings of 2^-24)."""
    import torch

    print(f"[head] N={N} V={V} ldw={ldw}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(V)
    W = torch.randn((2, ldw), generator=g, device="cuda")[:, :V]
    h = torch.randn((N, 2), generator=g, device="cuda")
    norm = torch.tensor([1.5, -0.5], device="cuda")
    got = H.rms_norm_lm_head(h, norm, W, 1e-5).double()
    a = h.double() * torch.rsqrt((h.double() ** 2).mean(1, keepdim=True) + 1e-5) * norm.double()
    assert bool(((got - a @ W.double()).abs() <= 1e-6 * (a.abs() @ W.double().abs())).all())


@pytest.mark.parametrize("N,D,V", [(40, 64, 70000), (40, 1000, 333), (100, 1016, 70001), (200, 1000, 50257)])
def test_a_nan_row_leaves_the_others_alone(N, D, V):
    """One broken row of hidden states: its logits are NaN, and no tile of the
    other rows is formed again (in another order of the sum: other bits)."""
    import torch

    print(f"[head] NaN row N={N} D={D} V={V}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(N)
    W = 0.02 * torch.randn((D, V), generator=g, device="cuda")
    h = torch.randn((N, D), generator=g, device="cuda")
    norm = torch.ones(D, device="cuda")
    ref = H.rms_norm_lm_head(h, norm, W, 1e-5).clone()
    for bad in (float("nan"), float("inf")):
        h[5, D // 2] = bad
        got = H.rms_norm_lm_head(h, norm, W, 1e-5)
        assert bool(got[5].isnan().all())
        got[5] = ref[5]
        assert torch.equal(got, ref)


# Every tile height in one and several slices, rows, k and columns all ragged.
TILES = [
    (45, 203, 50257, 64, 1),
    (45, 1015, 333, 64, 16),
    (100, 63, 70001, 128, 1),
    (100, 1015, 70001, 128, 2),
    (250, 203, 70001, 256, 1),
    (255, 1999, 20001, 256, 2),
]


@pytest.mark.parametrize("N,D,V,rows,slices", TILES)
def test_tile_plans(N, D, V, rows, slices):
    assert _plan(N, D, V) == (rows, slices)  # else this case tests another kernel than it names
    test_row_counts_and_edges(N, D, V)


@pytest.mark.parametrize("N,D,V,rows,slices", TILES)
def test_values_at_the_ends_of_float32_in_every_tile(N, D, V, rows, slices):
    assert _plan(N, D, V) == (rows, slices)
    test_values_at_the_ends_of_float32(N, D, V)


def test_tiny_rows_and_eps():
    """Rows of norm ~1e-3 (eps visible), an all-zero row (r = 1/sqrt(eps))."""
    h, norm, W = _case(3, 6, 96, 257, scale=1e-3)
    h[2] = 0.0
    got = H.rms_norm_lm_head(h, norm, W, 1e-5)
    ref = oracle.lm_head_logits(h, norm, W, 1e-5)
    bound = oracle.head_error_bound(h, norm, W, 1e-5)
    assert np.all(np.abs(got - ref) <= TOL * bound + 1e-30)
    assert np.all(got[2] == 0.0)


def test_strided_torch_buffers_and_full_size_against_torch():
    """h, lm_head and out as row-strided views (out a slice of a larger
    buffer, as the sampler's rotating logits sets are), at 256 x 4096 x
    128256, against torch's float32 product on the same device."""
    import torch

    torch.manual_seed(0)
    dev = torch.device("cuda:0")
    N, D, V = 256, 4096, 128256
    hbuf = torch.randn((N, D + 8), device=dev, dtype=torch.float32)
    h = hbuf[:, :D]
    norm = 1 + 0.1 * torch.randn(D, device=dev, dtype=torch.float32)
    W = 0.02 * torch.randn((D, V), device=dev, dtype=torch.float32)
    obuf = torch.full((N, V + 64), float("nan"), device=dev, dtype=torch.float32)
    out = obuf[:, :V]
    print("[head] full size 256x4096x128256", flush=True)
    H.rms_norm_lm_head(h, norm, W, 1e-5, out=out)
    torch.cuda.synchronize()
    assert torch.isnan(obuf[:, V:]).all(), "wrote past the row"
    r = torch.rsqrt((h.double() ** 2).mean(dim=1, keepdim=True) + 1e-5).float()
    a = (h * r) * norm
    ref = a @ W
    bound = a.abs().double() @ W.abs().double()
    err = (out.double() - ref.double()).abs()
    worst = float((err / bound).max())
    print(f"[head] worst error / bound {worst:.3e}", flush=True)
    assert worst <= TOL


def test_logits_stay_on_device_into_the_sampler():
    """LogitsHead output (a torch CUDA tensor) goes straight into
    sample_batch; ids equal the oracle's on the same logits (greedy rows
    exactly; sampled rows except draws within 1e-6 of a CDF boundary)."""
    from pagellm_amd.sampling import SamplingParams, sample_batch

    N, D, V = 12, 256, 32000
    h, norm, W = _case(11, N, D, V)
    head = H.LogitsHead(norm, W, 1e-5)
    logits = head(h)
    params = [SamplingParams(temperature=0.0)] * 4 + [SamplingParams(temperature=0.8, top_k=40)] * 4 + \
        [SamplingParams(temperature=1.0, top_p=0.9)] * 4
    u = np.random.default_rng(3).random(N)
    ids = sample_batch(logits, params, uniforms=u)
    host = logits.cpu().numpy()
    ref = oracle.sample_batch(host, params, u, None)
    for b in range(N):
        if ids[b] != ref[b]:
            assert b >= 4
            gap = oracle.draw_boundary_gap(oracle.probs(host[b], params[b], ()), u[b])
            cut = oracle.top_p_boundary_gap(host[b], params[b], ())
            assert gap < 1e-6 or cut < 1e-12, (b, gap, cut)
    bound = oracle.head_error_bound(h, norm, W, 1e-5)
    assert np.all(np.abs(host - oracle.lm_head_logits(h, norm, W, 1e-5)) <= TOL * bound + 1e-30)
