"""Bands at head_dims 8 to 128 on the MFMA kernels of flash_kernel.h, forward
and backward, against the oracle.

Lengths around the 16-row sub-tiles and 64-row tiles and blocks, head_dims
around the 32-column steps (padded columns, odd multiples of 8), windows
narrower and wider than a block, dilations and dense rows.  Tolerances: the
parity suites' (forward 1e-5 in fp32, gradients per check_grad); 16-bit forward
rows are rounded once from fp32 sums, so they lie within one unit of the last
place (2^-8 bf16, 2^-11 f16) plus 1e-4 for the rounding boundary.
"""
import numpy as np
import pytest
import torch

from conftest import check_grad, qkv, randn

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]

# N, D, left, right, dilation; left None: dense, causal when right == 0
SHAPES = [
    (1, 8, 3, 3, 1), (63, 16, 63, 0, 1), (64, 128, 127, 0, 1), (65, 32, 32, 31, 1), (130, 40, 5, 70, 1),
    (257, 96, 100, 17, 2), (300, 120, 200, 0, 3), (191, 72, 0, 64, 1), (513, 24, 16, 15, 1),
    (129, 128, None, 0, 1), (200, 80, None, 1, 1), (321, 32, None, 0, 1), (450, 128, None, 0, 1),
    # head_dim 64 (float32 on these kernels): windows past the stream kernels', causal rows in pairs of
    # tiles (an odd tile count, a ragged last one), dense rows
    (129, 64, 64, 64, 1), (700, 64, 100, 0, 2), (260, 64, 0, 127, 1), (64, 64, None, 0, 1), (65, 64, None, 0, 1),
    (330, 64, None, 0, 1), (257, 64, None, 1, 1),
]


@pytest.fixture(scope="module")
def ext():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import sparse_attention_cuda
    return sparse_attention_cuda


def _spec(oracle, shape, left, right, dil):
    if left is None:
        return oracle.Spec(*shape, pattern="dense", causal=right == 0)
    return oracle.Spec(*shape, pattern="sliding", left=left, right=right, dilation=dil)


# head_dim 64 in 16 bits runs on other kernels
CASES = [(*s, dt) for s in SHAPES for dt in DTYPES if s[1] != 64 or dt == torch.float32]


@pytest.mark.parametrize("N,D,left,right,dil,dtype", CASES)
def test_flash_against_oracle(ext, oracle, N, D, left, right, dil, dtype):
    shape = (2, N, 3, D)
    arrs = [*qkv(shape, 8000 + N + D), randn(shape, 8100 + N)]
    q, k, v, g = (torch.from_numpy(a).to(dtype).cuda() for a in arrs)
    up = [t.float().cpu().numpy() for t in (q, k, v, g)]
    spec = _spec(oracle, shape, left, right, dil)
    if left is None:
        y, grads = ext.dense_forward(q, k, v, right == 0), ext.dense_backward(q, k, v, g, right == 0)
    else:
        y, grads = ext.sliding_forward(q, k, v, left, right, dil), ext.sliding_backward(q, k, v, g, left, right, dil)
    ref = oracle.forward(spec, *up[:3])
    ulp = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    err = np.abs(y.float().cpu().numpy() - ref)
    assert (err <= (1e-5 if dtype == torch.float32 else 1e-4) + ulp * np.abs(ref)).all(), float(err.max())
    for name, a, b in zip("qkv", grads, oracle.backward(spec, *up)):
        check_grad("d" + name, a.float().cpu().numpy(), b, dtype == torch.float32)


@pytest.mark.parametrize("N,left,right,dil", [(64, 48, 1, 1), (129, 64, 64, 1), (700, 257, 0, 1), (321, 0, 49, 2),
                                               (1030, 300, 300, 1), (65, 1000, 0, 1), (500, 700, 200, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_flash_half_windows_at_64(ext, oracle, N, left, right, dil, dtype):
    """16-bit forward windows at head_dim 64 past the stream kernel's: each
    weight is rounded to 16 bits (by at most a part in 2^8 in bf16, 2^11 in f16,
    so that times sum p |v| bounds the row's error) and the row once more."""
    q, k, v = (torch.from_numpy(a).to(dtype).cuda() for a in qkv((2, N, 3, 64), 8800 + N))
    up = [t.float().cpu().numpy() for t in (q, k, v)]
    spec = _spec(oracle, (2, N, 3, 64), left, right, dil)
    y = ext.sliding_forward(q, k, v, left, right, dil).float().cpu().numpy()
    ref, mass = oracle.forward(spec, *up), oracle.forward(spec, *up[:2], np.abs(up[2]))
    u = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    err = np.abs(y - ref)
    assert (err <= 1e-4 + u * np.abs(ref) + u * mass).all(), float(err.max())


@pytest.mark.parametrize("N,H,left,right,G", [(300, 3, 129, 0, 16), (1100, 2, 200, 5, 3), (90, 2, 300, 0, 16),
                                              (12, 2, 200, 0, 16), (4300, 8, 131, 64, 1)])
def test_flash_wide_longformer(ext, oracle, N, H, left, right, G):
    """float32 Longformer windows past the stream kernel's ring: global rows
    from its partials, the others on the banded kernels (grids of 4 and 8
    waves), the window covering the globals, parted from them, and longer than
    the sequence; without a workspace the gather kernel.  The gradients run over
    split lists of the global tile and block."""
    import ma_attn as ma
    shape = (1, N, H, 64)
    arrs = [*qkv(shape, 8900 + N), randn(shape, 8910 + N)]
    q, k, v, g = (torch.from_numpy(a).cuda() for a in arrs)
    heads = sorted({0, H - 1})
    up = [np.ascontiguousarray(a[:, :, heads]) for a in arrs]
    spec = oracle.Spec(1, N, len(heads), 64, pattern="longformer", left=left, right=right, num_global=G)
    ref = oracle.forward(spec, *up[:3])
    gather = torch.empty_like(q)
    desc = ma.make_desc(*shape, ma.F32, ma.LONGFORMER, left=left, right=right, num_global=G)
    assert ma.workspace_size(desc) > 0
    ma.forward_raw(desc, q.data_ptr(), k.data_ptr(), v.data_ptr(), gather.data_ptr(), 0, 0,
                   torch.cuda.current_stream().cuda_stream)
    for y in (ext.longformer_forward(q, k, v, left, right, G), gather):
        assert float(np.abs(y.cpu().numpy()[:, :, heads] - ref).max()) <= 1e-5
    if N < 2000:
        grads = ext.longformer_backward(q, k, v, g, left, right, G)
        for name, x, y in zip("qkv", grads, oracle.backward(spec, *up)):
            check_grad("d" + name, x.cpu().numpy()[:, :, heads], y, True)


@pytest.mark.parametrize("N", [12, 32, 70, 96])
def test_longformer_float32_last_half_tile(ext, oracle, N):
    """float32 Longformer on the stream kernel with at least half of the last
    tile past the end, after a call that leaves NaN in LDS."""
    nan = torch.full((1, 256, 8, 64), float("nan"), device="cuda")
    arrs = qkv((1, N, 2, 64), 8960 + N)
    q, k, v = (torch.from_numpy(a).cuda() for a in arrs)
    ref = oracle.forward(oracle.Spec(1, N, 2, 64, pattern="longformer", left=0, right=0, num_global=5), *arrs)
    for _ in range(3):
        ext.longformer_forward(nan, nan, nan, 7, 0, 5)
        y = ext.longformer_forward(q, k, v, 0, 0, 5)
        assert float(np.abs(y.cpu().numpy() - ref).max()) <= 1e-5


def test_flash_wide_longformer_bad_values(ext):
    """A NaN key and value reach the rows that attend them and no others."""
    N, left, G, bad = 700, 150, 4, 300
    q, k, v = (torch.from_numpy(a).cuda() for a in qkv((1, N, 2, 64), 8950))
    want = ext.longformer_forward(q, k, v, left, 0, G)
    k[0, bad, 0] = v[0, bad, 0] = float("nan")
    got = ext.longformer_forward(q, k, v, left, 0, G)
    i = torch.arange(N, device="cuda")
    hit = (i < G) | ((i >= bad) & (i <= bad + left))
    assert bool(got[0, hit, 0].isnan().all())
    assert float((got[0, ~hit, 0] - want[0, ~hit, 0]).abs().max()) <= 1e-5
    assert torch.equal(got[0, :, 1], want[0, :, 1])
    q[0, 1, 1] = float("nan")  # a global row with no score that is a number
    got = ext.longformer_forward(q, k, v, left, 0, G)
    assert bool(got[0, 1, 1].isnan().all()) and torch.equal(got[0, 2:, 1], want[0, 2:, 1])


@pytest.mark.parametrize("N,H,causal", [(4200, 8, True), (9000, 16, True), (3000, 16, False)])
def test_flash_dense_grids(ext, oracle, N, H, causal):
    """float32 dense rows at head_dim 64 where the tiles pass one per CU (no
    pairs, 8 waves) and four per CU (two query groups per wave): sampled rows
    against the oracle."""
    shape = (1, N, H, 64)
    q, k, v = (torch.from_numpy(a).cuda() for a in qkv(shape, 8500 + N))
    y = ext.dense_forward(q, k, v, causal).cpu().numpy()
    up = [t.cpu().numpy()[:, :, [0, H - 1]] for t in (q, k, v)]
    ref = oracle.forward(oracle.Spec(1, N, 2, 64, pattern="dense", causal=causal), *up)
    assert float(np.abs(y[:, :, [0, H - 1]] - ref).max()) <= 1e-5


@pytest.mark.parametrize("B,N,H,causal", [(1, 300, 2, True), (1, 257, 2, False), (2, 4097, 3, True),
                                          (1, 8200, 16, True), (1, 4100, 16, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_flash_saved_statistics_half(ext, oracle, B, N, H, causal, dtype):
    """16-bit dense gradients at head_dim 64 from saved statistics on each
    grid: one row group per wave, pairs of tiles (2 x 3 heads of 4097 rows:
    198 128-row tiles), two row groups (16 heads); the first and last head
    against the oracle."""
    shape = (B, N, H, 64)
    arrs = [*qkv(shape, 8700 + N), randn(shape, 8710 + N)]
    q, k, v, g = (torch.from_numpy(a).to(dtype).cuda() for a in arrs)
    out, lse = ext.dense_forward(q, k, v, causal, return_lse=True)
    got = ext.dense_backward(q, k, v, g, causal, out=out, lse=lse)
    for b, h in ((0, 0), (B - 1, H - 1)):
        one = [np.ascontiguousarray(t[b:b + 1, :, h:h + 1].float().cpu().numpy()) for t in (q, k, v, g)]
        ref = oracle.backward(oracle.Spec(1, N, 1, 64, pattern="dense", causal=causal), *one)
        for name, x, y in zip("qkv", got, ref):
            check_grad("d" + name, x[b:b + 1, :, h:h + 1].float().cpu().numpy(), y, False)


@pytest.mark.parametrize("N,causal", [(300, True), (257, False), (65, True)])
def test_flash_saved_statistics(ext, oracle, N, causal):
    """float32 dense training pair at head_dim 64: the forward's statistics
    against a float64 log-sum-exp, and the gradients from them."""
    shape = (2, N, 3, 64)
    arrs = [*qkv(shape, 8600 + N), randn(shape, 8610 + N)]
    q, k, v, g = (torch.from_numpy(a).cuda() for a in arrs)
    out, lse = ext.dense_forward(q, k, v, causal, return_lse=True)
    s = torch.einsum("bihd,bjhd->bihj", q.double().cpu(), k.double().cpu()) / 8.0
    if causal:
        s = s.masked_fill(torch.arange(N)[None, :] > torch.arange(N)[:, None, None], float("-inf"))
    ref = torch.logsumexp(s, -1) / np.log(2.0)
    assert float((lse.double().cpu() - ref).abs().max()) <= 4e-6
    got = ext.dense_backward(q, k, v, g, causal, out=out, lse=lse)
    for name, a, b in zip("qkv", got, oracle.backward(oracle.Spec(*shape, pattern="dense", causal=causal), *arrs)):
        check_grad("d" + name, a.cpu().numpy(), b, True)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_flash_keeps_bad_values_to_their_rows(ext, dtype, bad):
    """An infinity or NaN in one key's V row reaches the queries that attend
    it and no other: the rest of the output, and the dK, dV rows that none of
    those queries attends, are as without it."""
    N, left, right, key = 200, 20, 7, 90
    arrs = [*qkv((1, N, 2, 96), 8300), randn((1, N, 2, 96), 8304)]
    q, k, v, g = (torch.from_numpy(a).to(dtype).cuda() for a in arrs)
    v2 = v.clone()
    v2[0, key, 1, 5] = bad
    y, y2 = (ext.sliding_forward(q, k, x, left, right) for x in (v, v2))
    sees = torch.zeros(N, dtype=torch.bool, device="cuda")
    sees[key - right:key + left + 1] = True  # query i attends [i - left, i + right]
    assert not torch.isfinite(y2[0, sees, 1, 5]).any()
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    torch.testing.assert_close(y2[0, ~sees], y[0, ~sees], rtol=tol, atol=tol)
    torch.testing.assert_close(y2[0, :, 0], y[0, :, 0], rtol=0, atol=0)  # the other head: untouched
    d1, d2 = (ext.sliding_backward(q, k, x, g, left, right) for x in (v, v2))
    far = torch.ones(N, dtype=torch.bool, device="cuda")
    far[key - right - left:key + left + right + 1] = False
    torch.testing.assert_close(d2[0][0, ~sees], d1[0][0, ~sees], rtol=tol, atol=tol)
    for a, b in zip(d2[1:], d1[1:]):
        torch.testing.assert_close(a[0, far], b[0, far], rtol=tol, atol=tol)


def test_flash_float32_extremes(ext):
    """float32 values near the largest finite one (above bf16's) and tiny ones
    pass through the three-plane products: one attended key gives O = V."""
    v = torch.tensor([3.4e38, -3.39e38, 1e-30, 3.0e38, -1e-20, 1.5, 3.3895314e38, -3.4028234e38], device="cuda")
    q = torch.zeros(1, 70, 1, 8, device="cuda")
    V = v.repeat(1, 70, 1, 1)
    o = ext.sliding_forward(q, q, V, 0, 0)
    torch.testing.assert_close(o, V, rtol=2e-7, atol=0)


def test_flash_launch_limit(ext):
    """2^24 one-row sequences: a workgroup each would pass a launch's 2^32
    threads, so the row kernels (4 rows a workgroup) keep this call.  One key
    has weight 1: O = V, dV = dO, dQ = dK = 0."""
    shape = (1 << 22, 1, 4, 40)
    q = torch.ones(shape, dtype=torch.bfloat16, device="cuda")
    v = torch.arange(1 << 24, device="cuda").remainder(251).to(torch.bfloat16).view(1 << 22, 1, 4, 1).expand(shape)
    v = v.contiguous()
    assert torch.equal(ext.sliding_forward(q, q, v, 3, 0), v)
    dq, dk, dv = ext.sliding_backward(q, q, q, v, 3, 0)
    assert torch.equal(dv, v)
    assert not dq.any() and not dk.any()


def _double(q, k, v, g, left, right):
    """Output and gradients of [1, N, 1, D] tensors in float64 (left None: every key)."""
    q, k, v, g = (t[0, :, 0].double().cpu() for t in (q, k, v, g))
    scale = q.shape[1] ** -0.5
    s = (q @ k.T) * scale
    if left is not None:
        d = torch.arange(len(q))[None, :] - torch.arange(len(q))[:, None]
        s = s.masked_fill((d < -left) | (d > right), float("-inf"))
    p = torch.softmax(s, -1)
    dp = g @ v.T
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * scale
    return p @ v, ds @ k, ds.T @ q, p.T @ g


@pytest.mark.parametrize("N,D", [(2048, 128), (2048, 32), (4096, 64)])
def test_flash_float32_long_rows(ext, N, D):
    """float32 rows of thousands of keys: a weight is off by its exponent's
    rounding, below 2^-20 for exponents down to -16, and a row's sums of N terms
    by about sqrt(N) 2^-25, so 2^-19 of each result's norm in all; an error per
    key block that adds up over a row (5e-6 and 1e-5 here) does not fit."""
    q, k, v, g = (torch.from_numpy(a).cuda() for a in [*qkv((1, N, 1, D), 8990 + D), randn((1, N, 1, D), 8991 + D)])
    got = [ext.dense_forward(q, k, v, False), *ext.dense_backward(q, k, v, g, False)]
    for name, x, ref in zip(("o", "dq", "dk", "dv"), got, _double(q, k, v, g, None, 0)):
        err = float((x[0, :, 0].cpu().double() - ref).norm() / ref.norm())
        print(f"  {name}: relative error {err:.2e}", flush=True)
        assert err <= 2.0 ** -19, name


@pytest.mark.parametrize("D", [16, 64])
@pytest.mark.parametrize("left,right", [(100, 20), (300, 300), (5000, 0)])
def test_flash_float32_window_error(ext, kernel_env, D, left, right):
    """float32 windows of hundreds of keys against float64: scores, weights'
    exponents (rounded at up to 2^-22, 2^-24 rms) and a sum rounded once per 32
    keys each come to under 2^-23 of the result's norm, and 2^-22 together; sums
    rounded six times per 32 keys, at 3.9e-7, do not fit."""
    kernel_env("MA_ATTN_KERNEL", "flash")
    N = 4096
    q, k, v = (torch.from_numpy(a).cuda() for a in qkv((1, N, 1, D), 8995 + D))
    y = ext.sliding_forward(q, k, v, left, right)[0, :, 0].cpu().double()
    ref = _double(q, k, v, q, left, right)[0]
    err = float((y - ref).norm() / ref.norm())
    print(f"  relative error {err:.2e}", flush=True)
    assert err <= 2.0 ** -22


# N, head_dim, left, right (left None: every key), dO's size, rows of dO 2^10 times as large
SMALL_GRADS = [(2048, 128, None, 0, 1e-3, None), (2048, 32, None, 0, 1e-3, None), (1500, 128, 600, 0, 1e-4, None),
               (700, 40, 100, 100, 1e-3, slice(400, 410)), (1000, 8, None, 0, 1.0, None)]


@pytest.mark.parametrize("N,D,left,right,size,loud", SMALL_GRADS)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_flash_half_keeps_small_weights(ext, N, D, left, right, size, loud, dtype):
    """16-bit calls at head_dims other than 64: the results of exact sums,
    rounded once, also where dS and P lie under f16's smallest steps (output
    gradients as an unscaled mean loss gives them, long rows).  A result is off
    by the rounding to the type, e, and by its float32 sums' f: the norms add
    in quadrature, and f up to 2^-18 of the result's norm moves the sum of
    bf16's e (2^-9.6) or f16's (2^-12.6) by less than one part in 2000.  A sum
    off by f of the elements' size lands on the other side of a rounding in
    about f 2^7 1.15 ln(1/f) of bf16's elements (spacing 2^-7 of the power of
    two below them, smaller elements more often): 1e-3 for the 5e-7 of sums of
    this length, 2.5e-3 and more where weights keep 16 bits."""
    q, k, v, g = (torch.from_numpy(a) for a in [*qkv((1, N, 1, D), 8970 + N), randn((1, N, 1, D), 8980 + N)])
    g *= size
    if loud is not None:
        g[:, loud] *= 1024
    q, k, v, g = (t.to(dtype).cuda() for t in (q, k, v, g))
    if left is None:
        got = [ext.dense_forward(q, k, v, False), *ext.dense_backward(q, k, v, g, False)]
    else:
        got = [ext.sliding_forward(q, k, v, left, right), *ext.sliding_backward(q, k, v, g, left, right)]
    for name, x, ref in zip(("o", "dq", "dk", "dv"), got, _double(q, k, v, g, left, right)):
        x = x[0, :, 0].cpu()
        err, store = float((x.double() - ref).norm()), float((ref.to(dtype).double() - ref).norm())
        flips = float((x != ref.to(dtype)).double().mean())
        print(f"  {name}: error {err:.4e}, of storing alone {store:.4e}, rounded otherwise {flips:.2e}", flush=True)
        assert err <= 1.0005 * store, name
        assert dtype == torch.float16 or flips <= 1.5e-3, name


@pytest.mark.parametrize("D", [24, 64, 128])
@pytest.mark.parametrize("dtype", DTYPES)
def test_flash_causal_rows_with_infinities(ext, dtype, D):
    """An infinity in the first key's V row makes that column of every causal
    row infinite and leaves the other columns alone; one in a query's dO makes
    that column of dV infinite, and dK infinite or NaN, for the keys it attends
    only."""
    N, r = 150, 70
    q, k, v, g = (torch.from_numpy(a).to(dtype).cuda()
                  for a in [*qkv((1, N, 2, D), 8400 + D), randn((1, N, 2, D), 8410)])
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    y = ext.dense_forward(q, k, v, True)
    v2 = v.clone()
    v2[0, 0, 1, 3] = float("inf")
    y2 = ext.dense_forward(q, k, v2, True)
    if D != 64 or dtype == torch.float32:  # 16-bit rows at head_dim 64 are another kernel's
        assert bool((y2[0, :, 1, 3] == float("inf")).all())
        y2[0, :, 1, 3] = y[0, :, 1, 3]
        torch.testing.assert_close(y2, y, rtol=tol, atol=tol)
    g2 = g.clone()
    g2[0, r, 1, 3] = float("inf")
    out, lse = ext.dense_forward(q, k, v, True, return_lse=True) if D == 64 else (None, None)
    d1, d2 = ([t.clone() for t in ext.dense_backward(q, k, v, x, True, out=out, lse=lse)] for x in (g, g2))
    assert not torch.isfinite(d2[0][0, r, 1]).any() and not torch.isfinite(d2[1][0, :r + 1, 1]).any()
    assert bool((d2[2][0, :r + 1, 1, 3] == float("inf")).all())
    d2[0][0, r, 1], d2[1][0, :r + 1, 1] = d1[0][0, r, 1], d1[1][0, :r + 1, 1]
    d2[2][0, :r + 1, 1, 3] = d1[2][0, :r + 1, 1, 3]
    for a, b in zip(d2, d1):
        torch.testing.assert_close(a, b, rtol=tol, atol=tol)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_flash_bad_values_cost(ext, dtype, D):
    """Calls in which every row is redone, as after an overflowed loss scale:
    at most 50 times the clean call's time (one wave per row, a key at a time,
    took 100 to 400 times).  NaN gradients leave the sums as they are."""
    N = 2048
    q, k, v, g = (torch.randn(1, N, 8, D, device="cuda").to(dtype) for _ in range(4))
    v2 = v.clone()
    v2[0, 0] = float("inf")

    def time(f):
        f()
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(3):
            f()
        b.record()
        b.synchronize()
        return a.elapsed_time(b)

    fwd, fwd2 = (time(lambda: ext.dense_forward(q, k, x, True)) for x in (v, v2))
    out, lse = ext.dense_forward(q, k, v, True, return_lse=True) if D == 64 else (None, None)
    bwd, bwd2, bwd3 = (time(lambda: ext.dense_backward(q, k, v, x, True, out=out, lse=lse))
                       for x in (g, torch.full_like(g, float("inf")), torch.full_like(g, float("nan"))))
    print(f"  forward {fwd2 / fwd:.1f}x, backward {bwd2 / bwd:.1f}x, NaN {bwd3 / bwd:.1f}x", flush=True)
    assert fwd2 <= 50 * fwd and bwd2 <= 50 * bwd and bwd3 <= 5 * bwd


# B, N, H, head_dim, left, right (left None: dense, causal when right == 0), dilation: both sides of every line of
# the dispatch between these kernels and the others, and classes that are shorter than the dilation
ROUTES = [
    *[(2, n, 3, D, 3, 3, 4) for n in (3, 8, 12, 17, 48, 52) for D in (16, 24, 48, 96)],
    *[(3, n, 2, D, 15, 0, 1) for n in (2, 4, 5, 12, 13) for D in (8, 48, 128)],
    *[(3, n, 2, D, None, 0, 1) for n in (2, 5, 13) for D in (16, 40, 128)],
    (1, 1000, 1, 96, 11, 12, 1), (1, 1000, 1, 96, 12, 12, 1), (1, 500, 1, 80, 10, 11, 1), (1, 4001, 1, 72, 1, 1, 1),
    (1, 2001, 1, 128, 0, 0, 1), (1, 2000, 1, 16, 3, 3, 1), (1, 2001, 1, 32, 3, 3, 2), (2, 30, 2, 48, 40, 40, 100),
    *[(2, n, 2, 64, 300, 300, 4) for n in (5, 96, 100, 130)], (2, 64, 2, 64, 64, 64, 1), (2, 65, 2, 64, 64, 64, 1),
    (1, 4032, 8, 64, 64, 64, 1), (1, 4096, 8, 64, 40, 30, 1), (5, 40, 2, 64, 100, 0, 64), (1, 129, 2, 64, 100, 100, 1),
    *[(2, n, 2, 64, None, 0, 1) for n in (32, 33, 64, 128, 129, 256, 257)],
    *[(2, n, 2, 64, None, 1, 1) for n in (32, 65, 129)], (257, 64, 2, 64, None, 0, 1), (129, 129, 1, 64, None, 1, 1),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_flash_routes_agree(ext, kernel_env, dtype):
    """The call as dispatched, on these kernels wherever they can take it, and
    on none of them: float32 within the parity suites' tolerance, bf16 within two
    roundings (2^-7) and, at head_dim 64, weights of 16 bits."""
    tol = dict(rtol=1e-5, atol=2e-5) if dtype == torch.float32 else dict(rtol=2.0 ** -7, atol=2e-2)
    for i, (B, N, H, D, left, right, dil) in enumerate(ROUTES):
        gen = torch.Generator(device="cuda").manual_seed(i)
        q, k, v, g = (torch.randn(B, N, H, D, generator=gen, device="cuda").to(dtype) for _ in range(4))
        got = {}
        for route in ("default", "flash", "noflash"):
            kernel_env("MA_ATTN_KERNEL", route)
            if left is None:
                got[route] = [ext.dense_forward(q, k, v, right == 0), *ext.dense_backward(q, k, v, g, right == 0)]
                if D == 64:
                    out, lse = ext.dense_forward(q, k, v, right == 0, return_lse=True)
                    got[route] += ext.dense_backward(q, k, v, g, right == 0, out=out, lse=lse)
            else:
                got[route] = [ext.sliding_forward(q, k, v, left, right, dil),
                              *ext.sliding_backward(q, k, v, g, left, right, dil)]
        for route in ("flash", "noflash"):
            for x, y in zip(got["default"], got[route]):
                torch.testing.assert_close(x, y, **tol, msg=lambda m: f"{ROUTES[i]} {route}: {m}")


@pytest.mark.parametrize("N,D,left,right,dil", [(129, 64, 64, 64, 1), (700, 64, 100, 0, 2), (257, 64, None, 1, 1),
                                               (100, 96, 3, 3, 1), (65, 48, 2, 9, 8), (12, 128, None, 0, 1),
                                               (190, 64, None, 0, 1), (30, 64, 20, 70, 3)])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("route", ["flash", "noflash"])
def test_flash_forced_routes(ext, oracle, kernel_env, route, N, D, left, right, dil, dtype):
    """Small calls on these kernels though others are faster for them, and on the
    others (per-tile and row kernels that the dispatch reaches only for rows
    past 2^31 bytes or 2^24 tiles), against the oracle."""
    kernel_env("MA_ATTN_KERNEL", route)
    shape = (2, N, 3, D)
    arrs = [*qkv(shape, 8200 + N), randn(shape, 8210 + N)]
    q, k, v, g = (torch.from_numpy(a).to(dtype).cuda() for a in arrs)
    up = [t.float().cpu().numpy() for t in (q, k, v, g)]
    spec, extra = _spec(oracle, shape, left, right, dil), []
    if left is None:
        y, grads = ext.dense_forward(q, k, v, right == 0), ext.dense_backward(q, k, v, g, right == 0)
        if D == 64:
            out, lse = ext.dense_forward(q, k, v, right == 0, return_lse=True)
            extra = ext.dense_backward(q, k, v, g, right == 0, out=out, lse=lse)
    else:
        y, grads = ext.sliding_forward(q, k, v, left, right, dil), ext.sliding_backward(q, k, v, g, left, right, dil)
    ref, want = oracle.forward(spec, *up[:3]), oracle.backward(spec, *up)
    u = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    mass = oracle.forward(spec, *up[:2], np.abs(up[2])) if D == 64 else 0.0  # weights of 16 bits there
    err = np.abs(y.float().cpu().numpy() - ref)
    assert (err <= (1e-5 if dtype == torch.float32 else 1e-4) + u * np.abs(ref) + u * mass).all(), float(err.max())
    for name, a, b in zip(("dq", "dk", "dv") * 2, [*grads, *extra], [*want, *want]):
        check_grad(name, a.float().cpu().numpy(), b, dtype == torch.float32)


@pytest.mark.parametrize("N,left,right,dil", [(64, 32, 31, 1), (130, 100, 0, 1), (300, 70, 70, 2), (65, 300, 9, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_band_kernel(ext, oracle, kernel_env, N, left, right, dil, dtype):
    """16-bit windows at head_dim 64 on the band kernel (rows past the others'
    2^31 bytes): weights and rows rounded to 16 bits."""
    kernel_env("MA_ATTN_KERNEL", "band")
    q, k, v = (torch.from_numpy(a).to(dtype).cuda() for a in qkv((2, N, 3, 64), 8250 + N))
    up = [t.float().cpu().numpy() for t in (q, k, v)]
    spec = _spec(oracle, (2, N, 3, 64), left, right, dil)
    y = ext.sliding_forward(q, k, v, left, right, dil).float().cpu().numpy()
    ref, mass = oracle.forward(spec, *up), oracle.forward(spec, *up[:2], np.abs(up[2]))
    u = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    err = np.abs(y - ref)
    assert (err <= 1e-4 + u * np.abs(ref) + u * mass).all(), float(err.max())


# calls that 64-row tiles served 2 to 6 times slower than the kernels before them
SHORT = [(64, 256, 4, 64, 300, 300, 64, False), (64, 10, 4, 48, 3, 3, 7, False), (64, 10, 4, 128, 3, 3, 7, True),
         (1024, 2, 4, 128, None, 0, 1, False), (512, 64, 4, 64, None, 1, 1, False), (1, 300, 1, 128, 3, 3, 1, False)]


@pytest.mark.parametrize("B,N,H,D,left,right,dil,backward", SHORT)
def test_flash_dispatch_short_calls(ext, kernel_env, B, N, H, D, left, right, dil, backward):
    """Short classes and small grids in float32 take no more than 1.5 times the
    time of the other kernels (20 calls in a graph)."""
    q, k, v, g = (torch.randn(B, N, H, D, device="cuda") for _ in range(4))

    def call():
        if left is None:
            return ext.dense_backward(q, k, v, g, right == 0) if backward else ext.dense_forward(q, k, v, right == 0)
        return ext.sliding_backward(q, k, v, g, left, right, dil) if backward else \
            ext.sliding_forward(q, k, v, left, right, dil)

    def time():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            call()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(20):
                call()
        graph.replay()
        times = []
        for _ in range(3):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            graph.replay()
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    t = time()
    kernel_env("MA_ATTN_KERNEL", "noflash")
    other = time()
    print(f"  {50 * t:.1f} us, other kernels {50 * other:.1f}", flush=True)
    assert t <= 1.5 * other


def test_flash_launch_limit_forced(ext, kernel_env):
    """As test_flash_launch_limit, with the banded kernels asked for: the limit,
    not the length of the sequences, leaves the call to the row kernels."""
    kernel_env("MA_ATTN_KERNEL", "flash")
    test_flash_launch_limit(ext)
