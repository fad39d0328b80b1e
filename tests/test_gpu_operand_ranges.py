"""Operands of unusual scale through the entry points whose arithmetic is fp32 (fused, tiled, naive).

fp32 arithmetic holds every weight and value to 24 bits of itself, whatever stands beside it: a small
column of V, a small probability, a value near the largest float, an infinity. The kernels that take
operands in 16-bit terms or sum before they normalise are held to that here.
"""
import math

import pytest
import torch

import cuda_attn
from cuda_attn import _native
from cuda_attn.workloads import make_qkv

pytestmark = pytest.mark.gpu

F32, F16 = torch.float32, torch.float16
INF = float("inf")
# Grids of each form of fused with fp32 inputs: the fp32 matrix core, two key groups, one key group.
FUSED_F32_GRIDS = [(3, 300), (60, 300), (300, 300), (8, 4096), (80, 1024)]


def reference64(q, k, v, causal=False):
    """float64 softmax(QK^T/sqrt(d))V of the visible keys (a head at a time; V may hold infinities)."""
    b, h, n, d = q.shape
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for i in range(b):
        for j in range(h):
            s = torch.matmul(q[i, j].double(), k[i, j].double().t().contiguous()) / math.sqrt(d)
            if causal:
                s.masked_fill_(torch.ones_like(s, dtype=torch.bool).triu(1), -INF)
            out[i, j] = torch.matmul(torch.softmax(s, -1), v[i, j].double())
    return out


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("bh,n", FUSED_F32_GRIDS)
def test_fused_fp32_column_scales(bh, n, large, causal):
    """Columns of V of very different scales beside each other (and on both sides of 2^-20): an output
    column depends on its own column of V alone, so its relative error does not depend on the scale.
    4e-6 in the 2-norm per head and column (fp32 sums are seen 2e-7 to 1.2e-6 off)."""
    q, k, v = make_qkv(1, bh, n, 64, F32, seed=17, device="cuda")
    scale = torch.ones(64, device="cuda")
    scale[8:16] = torch.tensor([1.0, 2.0 ** -17, 2.0 ** -20, 2.0 ** -23, 1e-8, 1e-10, 1e-12, 1e-14])
    scale[20], scale[30] = 1e-20, 1e-30
    if large:
        scale[21], scale[40] = 1e4, 1e25
    v = v * scale
    heads = list(range(0, bh, max(1, bh // 4)))
    out = cuda_attn.fused(q, k, v, causal)[:, heads].double()
    ref = reference64(q[:, heads], k[:, heads], v[:, heads], causal)
    err = torch.linalg.vector_norm(out - ref, dim=2) / torch.linalg.vector_norm(ref, dim=2)
    assert err.max().item() <= 4e-6


@pytest.mark.parametrize("name,dtype,bh,n", [("fused", F32, *g) for g in FUSED_F32_GRIDS] +
                         [("fused", F16, *g) for g in ((2, 300), (300, 320), (300, 200), (140, 1000), (300, 40))] +
                         [("tiled", dt, *g) for dt in (F32, F16) for g in ((2, 300), (64, 515))])
def test_causal_rows_do_not_see_later_tokens(name, dtype, bh, n):
    """Causal rows keep their bits when only later tokens change, to scores and values of another scale."""
    q, k, v = make_qkv(1, bh, n, 64, dtype, seed=19, device="cuda")
    out = getattr(cuda_attn, name)(q, k, v, True)
    for j in (n // 2 + 5, n - 3):
        k2, v2 = k.clone(), v.clone()
        k2[:, :, j:] *= 500
        v2[:, :, j:] *= 1e9 if dtype == F32 else 1e3
        same = torch.equal(getattr(cuda_attn, name)(q, k2, v2, True)[:, :, :j], out[:, :, :j])
        assert same, j


@pytest.mark.parametrize("bh,n", FUSED_F32_GRIDS)
def test_fused_fp32_single_products(bh, n):
    """Scores of a single product each (one nonzero dim in Q): no sum averages the operands' roundings.
    Three roundings of fp32 of a score in the log2 domain (|x| <= X) put a probability off by at most
    ln 2 * 3 * 2^-24 X, an output by twice that of the largest |V|, and 2e-6 for the other steps."""
    q, k, v = make_qkv(1, bh, n, 64, F32, seed=23, device="cuda")
    q[..., :11] = 0
    q[..., 12:] = 0
    q[..., 11] *= 30
    k[..., 11] *= 4
    heads = list(range(0, bh, max(1, bh // 4)))
    out = cuda_attn.fused(q, k, v)[:, heads].double()
    ref = reference64(q[:, heads], k[:, heads], v[:, heads])
    x = (q[..., 11].abs() / 8 * 1.4427)[:, heads].unsqueeze(-1) * k[..., 11].abs()[:, heads].amax(-1)[..., None, None]
    bound = (2 * math.log(2) * 3 * 2.0 ** -24 * x + 2e-6) * v.abs().max()
    assert bool(((out - ref).abs() <= bound).all())


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("bh,n,d", [(1, 2, 64), (3, 333, 40), (2, 130, 128), (70, 515, 64), (40, 901, 96)])
def test_tiled_fp32_largest_values(bh, n, d, causal):
    """Values near the largest float, which a sum of unnormalised weights would carry to infinity."""
    q, k, v = make_qkv(1, bh, n, d, F32, seed=29, device="cuda")
    v = 3.2e38 * (1 - 0.05 * v.abs().clamp(max=10) / 10) * torch.where(torch.arange(d, device="cuda") % 3 == 0, -1.0, 1.0)
    v[..., 1] = torch.randn(v.shape[:-1], device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    heads = list(range(0, bh, max(1, bh // 4)))
    out = cuda_attn.tiled(q, k, v, causal)[:, heads].double()
    ref = reference64(q[:, heads], k[:, heads], v[:, heads], causal)
    big = torch.arange(d, device="cuda") != 1
    assert bool(((out - ref)[..., big].abs() <= 4e-6 * ref[..., big].abs()).all())
    assert bool(((out - ref)[..., 1].abs() <= 1e-5).all())


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [F16, F32])
@pytest.mark.parametrize("bh,n,d", [(2, 37, 40), (2, 300, 64), (3, 301, 80), (2, 131, 128), (64, 515, 64), (64, 514, 40),
                                    (64, 513, 128)])
def test_tiled_infinite_values(bh, n, d, dtype, causal):
    """An infinite element of V is infinite in its dim of the rows that see it, a NaN is NaN there, and
    nothing else is touched."""
    q, k, v = make_qkv(1, bh, n, d, dtype, seed=31, device="cuda")
    places = {(0, n // 2, 5): INF, (0, n // 3, 7): -INF, (bh - 1, n - 1, 33): INF, (bh - 1, 2, 34): float("nan")}
    zeroed = v.clone()
    for (h, key, c), x in places.items():
        v[0, h, key, c], zeroed[0, h, key, c] = x, 0
    out, want = cuda_attn.tiled(q, k, v, causal), cuda_attn.tiled(q, k, zeroed, causal)
    rows = torch.arange(n, device="cuda")
    keep = torch.ones_like(out, dtype=torch.bool)
    for (h, key, c), x in places.items():
        sees = rows >= key if causal else rows >= 0
        got = out[0, h, sees, c]
        assert bool(got.isnan().all() if math.isnan(x) else (got == x).all())
        keep[0, h, sees, c] = False
    bar = 1e-5 if dtype == F32 else 2e-3
    assert bool(((out - want).abs()[keep] <= bar).all())


# Key split, persistent with whole and ragged last tiles, one tile a row.
FUSED_F16_GRIDS = [(2, 300), (300, 320), (300, 200), (140, 1000), (3, 64), (300, 40)]


@pytest.mark.parametrize("out_dtype", [F16, F32])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("bh,n", FUSED_F16_GRIDS)
def test_fused_fp16_infinite_value_of_small_weight(bh, n, causal, out_dtype):
    """An infinite element of V whose key has a weight of e^-50 (any positive fp32 weight makes it
    infinite), in the key groups and launch forms of fused with fp16 inputs."""
    q, k, v = make_qkv(1, bh, n, 64, F16, seed=37, device="cuda")
    q[..., 0] = 1
    j = min(17, n - 2)
    k[..., 0] = 0
    k[..., j, :] = 0
    k[..., j, 0] = -400
    want = cuda_attn.fused(q, k, v, causal, out_dtype=out_dtype)
    v[0, 0, j, 5] = INF
    v[0, bh - 1, j, 63] = -INF
    rows = torch.arange(n, device="cuda")
    sees = rows > j if causal else rows >= 0
    for persistent in (True, False):
        prev = _native.set_persistent(persistent)
        try:
            out = cuda_attn.fused(q, k, v, causal, out_dtype=out_dtype)
        finally:
            _native.set_persistent(prev)
        assert bool((out[0, 0, sees, 5] == INF).all() and (out[0, bh - 1, sees, 63] == -INF).all())
        keep = torch.ones_like(out, dtype=torch.bool)
        keep[0, 0, :, 5] = keep[0, bh - 1, :, 63] = False
        same = torch.equal(out[keep], want[keep])
        assert same
        hidden = rows < j if causal else rows < 0
        assert bool(((out - want)[:, :, hidden].abs() <= 2e-3).all())


def one_hot_weights(bh, n, dtype, seed, value=1.0):
    """Integer q and k (exact dot products, scores with a standard deviation of 4) and a V that shows
    the weights of 64 keys, spread over the row, one a dim."""
    g = torch.Generator().manual_seed(seed)
    q, k = (torch.randint(-3, 4, (1, bh, n, 64), generator=g).to(dtype).cuda() for _ in range(2))
    v = torch.zeros(1, bh, n, 64, dtype=dtype, device="cuda")
    keys = torch.arange(64, device="cuda") * n // 64
    v[:, :, keys, torch.arange(64, device="cuda")] = value
    return q, k, v


@pytest.mark.parametrize("bh,n", [(2, 64), (2, 300), (300, 320), (300, 200), (140, 1000)])
def test_fused_fp16_small_weights(bh, n):
    """Each weight of fused with fp16 inputs (fp32 output) against float64, relative to itself: an
    exponent of up to 64 is rounded at 2^-19 with 2^-26 of it in the scale (ln 2 of the two: 2e-6),
    2^x, the terms and the division add 2^-22 each; below that, an absolute 2^-42 of the row's largest."""
    q, k, v = one_hot_weights(bh, n, F16, seed=41)
    heads = list(range(0, bh, max(1, bh // 4)))
    out = cuda_attn.fused(q, k, v, out_dtype=F32)[:, heads].double()
    ref = reference64(q[:, heads], k[:, heads], v[:, heads])
    assert bool(((out - ref).abs() <= 4e-6 * ref + 2.0 ** -42).all())


@pytest.mark.parametrize("name,bh,n", [("fused", 2, 64), ("fused", 2, 300), ("fused", 300, 320), ("fused", 140, 1000),
                                       ("tiled", 2, 64), ("tiled", 3, 301), ("tiled", 64, 516), ("tiled", 140, 1000)])
def test_fp16_small_weights_of_large_values(name, bh, n):
    """fp16 in and out with 60000 at the key whose weight a dim shows: the products of weights down to
    2^-41 round to what fp32 arithmetic gives: half an ulp of fp16 (2^-11 of it, 2^-25 below the normal
    range), the weight's own error, and 60000 times an absolute 2^-43 of the row's largest weight."""
    q, k, v = one_hot_weights(bh, n, F16, seed=43, value=60000.0)
    heads = list(range(0, bh, max(1, bh // 4)))
    out = getattr(cuda_attn, name)(q, k, v)[:, heads].double()
    ref = reference64(q[:, heads], k[:, heads], v[:, heads])
    assert bool(((out - ref).abs() <= (2.0 ** -11 + 8e-6) * ref + 2.0 ** -25 + 6e4 * 2.0 ** -43).all())
