"""fp32 GEMM on split bf16 operands (csrc/gemm_split.hip) against float64.

Tolerance: each of the K products is rounded once (2^-24) and K / 16 partial
sums are accumulated in fp32, in six passes; a random walk of 6 K / 16 roundings
of the running sum stays below 2^-24 sqrt(6 K / 16) of |a| |w| per element, and
four times that bounds the largest of 10^6 elements.
"""

import math

import pytest
import torch

from cutilegpt_amd import _lib

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32


def run(gpu, a, w, b, epi, out_dtype=F32, tile=_lib.TILE_AUTO, c=None):
    m, k = a.shape
    n = w.shape[0]
    out = torch.empty((m, n), dtype=out_dtype, device=gpu) if c is None else c.clone()
    code = _lib.CGPT_F32 if out_dtype == F32 else _lib.CGPT_BF16
    _lib.check(_lib.load().cgpt_gemm(
        a.data_ptr(), w.data_ptr(), None if b is None else b.data_ptr(), out.data_ptr(), m, n, k,
        a.stride(0), w.stride(0), out.stride(0), _lib.CGPT_F32, _lib.CGPT_F32, code, epi, tile,
        torch.cuda.current_stream(gpu).cuda_stream), "gemm")
    return out


def randn(gpu, *shape, seed=0, scale=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).to(gpu)


def check(out, a, w, ref):
    k = a.shape[1]
    scale = a.double().norm(dim=1)[:, None] * w.double().norm(dim=1)[None, :] + 1.0
    tol = 4 * 2.0 ** -24 * math.sqrt(6 * k / 16 + 16)
    err = ((out.double() - ref).abs() / scale).max().item()
    assert err <= tol, (err, tol)


# One or more shapes for each tile of the size rule, at the edges of tiles and
# of the 16-wide k stages (whole, partial, fewer than the K groups).
SHAPES = [
    (65, 1, 4), (65, 33, 20), (97, 31, 64), (87, 768, 3072),           # 32x32, 8 groups
    (300, 1000, 36), (65, 3072, 768),                                  # 32x32, 4 groups
    (193, 3000, 52), (200, 3072, 768),                                 # 64x64, 4 groups
    (513, 3100, 100), (520, 3072, 768),                                # 128x64, 2 groups
    (1409, 1537, 1540), (1500, 1600, 1600),                            # 128x128, 2 groups
    (2049, 5121, 44), (87, 50257, 64),                                 # 128x128
    (16, 130, 512), (17, 130, 512), (17, 130, 508), (33, 130, 252),    # 64 rows or fewer: the skinny
    (33, 131, 256), (64, 4800, 1600), (32, 16384, 512), (33, 16385, 512),  # kernel or a split tile
    (4095, 4100, 28), (4096, 6144, 80),                                # 256x256
]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_split_shapes(gpu, m, n, k):
    a, w, b = randn(gpu, m, k, seed=1), randn(gpu, n, k, seed=2), randn(gpu, n, seed=3)
    ref = a.double() @ w.double().t() + b.double()
    check(run(gpu, a, w, b, _lib.EPI_BIAS), a, w, ref)
    c = randn(gpu, m, n, seed=4)
    check(run(gpu, a, w, b, _lib.EPI_BIAS_RESID, c=c), a, w, ref + c.double())


@pytest.mark.parametrize("tile", [0, 1, _lib.TILE_AUTO])
def test_split_epilogues_strides_bf16_out(gpu, tile):
    m, n, k = 130, 70, 76
    a = randn(gpu, m, k + 8, seed=1)[:, 4:4 + k]  # lda 84, 16-byte aligned rows
    w, b = randn(gpu, n, k, seed=2, scale=0.2), randn(gpu, n, seed=3)
    ref = a.double() @ w.double().t()
    check(run(gpu, a, w, None, _lib.EPI_NONE, tile=tile), a, w, ref)
    g = torch.nn.functional.gelu(ref + b.double(), approximate="tanh")
    check(run(gpu, a, w, b, _lib.EPI_BIAS_GELU, tile=tile), a, w, g)
    out = run(gpu, a, w, b, _lib.EPI_BIAS, BF16, tile=tile)
    assert ((out.double() - ref - b.double()).abs() <= 2.0 ** -8 * (ref + b.double()).abs() + 1e-5).all()


@pytest.mark.parametrize("m,n,k", [(130, 70, 40), (300, 1000, 36), (700, 2100, 48), (2049, 5121, 32)])
def test_split_non_finite(gpu, m, n, k):
    """Infinities and NaN in either operand, values that round to infinity in
    bf16 (finite in fp32), and overflowing sums give fp32's results."""
    a, w, b = randn(gpu, m, k, seed=1), randn(gpu, n, k, seed=2), randn(gpu, n, seed=3)
    a[3, 5], a[70, 1], w[60, 2], w[61, 3] = math.inf, math.nan, -math.inf, math.nan
    w[5] = 0.0
    w[5, 6] = 1.0                    # inf * 0 only at k = 5: column 5 of row 3 is NaN
    a[100, 7] = 3.4e38               # rounds to infinity in bf16
    w[:, 7] *= 1e-3
    # One product past fp32's range (float64 holds it, so the reference only
    # agrees if no other sum of row 101 or column 9 leaves fp32's range by
    # itself: |0.1 x| 3e38 <= 1.5e38 for |x| <= 5).
    a[:, 0] *= 0.1
    w[:, 0] *= 0.1
    a[101, 0], w[9, 0] = 3e38, 3e38
    ref = (a.double() @ w.double().t() + b.double()).float()
    out = run(gpu, a, w, b, _lib.EPI_BIAS)
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(torch.isinf(out), inf) and torch.equal(out[inf], ref[inf])
    fin = torch.isfinite(ref)
    scale = (a.double().nan_to_num(0, 0, 0).norm(dim=1)[:, None] *
             w.double().nan_to_num(0, 0, 0).norm(dim=1)[None, :] + 1.0)
    assert ((out.double() - ref.double()).abs()[fin] / scale[fin]).max() < 1e-6


@pytest.mark.parametrize("scale", [1e-28, 1e-31, 1e-36, 1e-38])
def test_split_tiny_rows(gpu, scale):
    """Rows too small for three bf16 parts keep fp32's precision."""
    m, n, k = 100, 90, 64
    a, w = randn(gpu, m, k, seed=1), randn(gpu, n, k, seed=2)
    a[::3] *= scale
    w[::2] *= 1e6
    ref = a.double() @ w.double().t()
    out = run(gpu, a, w, None, _lib.EPI_NONE)
    row = (out.double() - ref).norm(dim=1) / ref.norm(dim=1)
    # Products of subnormal results carry absolute errors of 2^-149 each.
    assert row.max() < 4 * 2.0 ** -24 * math.sqrt(k), row.max()


# A shape for each tile of the size rule, K past the fp32 MFMA kernel's and ending
# within a stage.
TILES = [(65, 33, 68), (2700, 192, 132), (300, 1000, 84), (1500, 384, 76), (1500, 768, 84), (100, 38400, 72),
         (2049, 5121, 76), (1409, 1537, 1540), (4090, 4092, 84)]


# 33 to 64 rows on either side of the skinny kernel's band of N.
@pytest.mark.parametrize("m,n,k", [(33, 4096, 256), (33, 4100, 256), (64, 8192, 260), (48, 8196, 260),
                                   (49, 4104, 1600), (49, 4104, 1596)])
def test_skinny_band(gpu, m, n, k):
    test_split_shapes(gpu, m, n, k)


@pytest.mark.parametrize("m,n,k", TILES)
def test_split_tiles(gpu, m, n, k):
    test_split_shapes(gpu, m, n, k)


@pytest.mark.parametrize("m,n,k", TILES)
def test_split_tiles_non_finite(gpu, m, n, k):
    """A NaN, infinities and values past the split's range, in single rows."""
    a, w, b = randn(gpu, m, k, seed=1), randn(gpu, n, k, seed=2), randn(gpu, n, seed=3)
    a[m - 1, k - 1], a[m // 2, 3], w[n - 1, k - 2] = math.nan, math.inf, -math.inf
    a[3, 5] = 3.4e38
    w[:, 5] *= 1e-3
    ref = (a.double() @ w.double().t() + b.double()).float()
    out = run(gpu, a, w, b, _lib.EPI_BIAS)
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(out[inf], ref[inf])
    fin = torch.isfinite(ref)
    size = a.double().nan_to_num(0, 0, 0).abs() @ w.double().nan_to_num(0, 0, 0).abs().t() + 1.0
    assert ((out.double() - ref.double()).abs()[fin] / size[fin]).max() < 1e-6


# The fp32 MFMA kernel of short K, at the edges of its rule, its tiles (64x64,
# 128x128 from 512 of them) and 4-wide stores, and for rows 2^22 apart.
@pytest.mark.parametrize("m,n,k", [(1, 1, 4), (16, 130, 64), (65, 33, 44), (65, 64, 16), (520, 577, 48),
                                   (1025, 301, 60), (4095, 2051, 64), (8191, 1153, 32), (100, 50257, 20)])
def test_short_k(gpu, m, n, k):
    test_split_shapes(gpu, m, n, k)
    a, w, b = randn(gpu, m, k, seed=1), randn(gpu, n, k, seed=2, scale=0.2), randn(gpu, n, seed=3)
    ref = a.double() @ w.double().t() + b.double()
    check(run(gpu, a, w, b, _lib.EPI_BIAS_GELU), a, w, torch.nn.functional.gelu(ref, approximate="tanh"))
    out = run(gpu, a, w, b, _lib.EPI_BIAS, BF16)
    assert ((out.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5).all()


@pytest.mark.parametrize("epi", [_lib.EPI_BIAS, _lib.EPI_BIAS_RESID])
def test_rows_far_apart(gpu, epi):
    m, n, k = 70, 90, 100
    a = torch.empty(70, 1 << 22, device=gpu)[:, :k]
    a.copy_(randn(gpu, m, k, seed=1))
    w, b, c = randn(gpu, n, k, seed=2), randn(gpu, n, seed=3), randn(gpu, m, n, seed=4)
    ref = a.double() @ w.double().t() + b.double() + (c.double() if epi == _lib.EPI_BIAS_RESID else 0)
    check(run(gpu, a, w, b, epi, c=c), a, w, ref)


# Small elements in rows that hold ordinary ones too, each against a partner of
# the inverse scale; e < 0: in W.  Products are of order one, so the bound of
# `check` holds with the sum of their sizes for the norms.
@pytest.mark.parametrize("e", [-125, -115, -100, -80, 80, 100, 106, 115, 125])
@pytest.mark.parametrize("m,n,k", TILES + [(300, 1000, 36)])
def test_split_inverse_scales(gpu, m, n, k, e):
    a, w = randn(gpu, m, k, seed=1), randn(gpu, n, k, seed=2)
    a[:, 1::2] *= 2.0 ** -e
    w[:, 1::2] *= 2.0 ** e
    w[:, 0] = 0.0                    # nothing large against the ordinary a[:, 0]
    ref = a.double() @ w.double().t()
    size = a.double().abs() @ w.double().abs().t()
    out = run(gpu, a, w, None, _lib.EPI_NONE)
    tol = 4 * 2.0 ** -24 * math.sqrt(6 * k / 16 + 16)
    assert ((out.double() - ref).abs() / size).max() <= tol


@pytest.mark.parametrize("scale", [1e-38, 1e-42, 1e-44])
def test_split_smallest_values(gpu, scale):
    """Small and subnormal values beside ordinary ones that meet zeros."""
    m, n, k = 100, 90, 72
    a, w = randn(gpu, m, k, seed=1), randn(gpu, n, k, seed=2) * 1e30
    a[:, ::2] *= scale
    w[:, 1::2] = 0.0
    ref = a.double() @ w.double().t()
    size = a.double().abs() @ w.double().abs().t()
    out = run(gpu, a, w, None, _lib.EPI_NONE)
    assert ((out.double() - ref).abs() / size).max() <= 4 * 2.0 ** -24 * math.sqrt(k)
