"""16-bit GEMM with K shared between wave groups (csrc/gemm_kgroup.hip), as
TILE_AUTO picks it for problems of few tiles, against float64.

Shapes: for each of its tiles the edges of rows and columns, K of one k64 stage
(fewer than the groups), a stage count the groups do not divide, and the largest
M of the tile's range."""

import math

import pytest
import torch

from cutilegpt_amd import _lib

pytestmark = pytest.mark.gpu
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32
CODE = {BF16: _lib.CGPT_BF16, F16: _lib.CGPT_F16, F32: _lib.CGPT_F32}

SHAPES = [
    (65, 36, 64), (70, 100, 128), (97, 768, 3072), (130, 260, 192),   # 32x32, 4 groups
    (300, 900, 320), (591, 768, 3072),                                # 64x32, 4 groups
    (1000, 768, 768), (1100, 772, 1088),                              # 64x64, 2 groups
    (1500, 768, 3072),                                                # 64x96, 2 groups
    (2700, 768, 768), (2690, 764, 832),                               # 96x96, 2 groups
    (2900, 772, 704), (3300, 768, 3072),                              # 128x96
    (2048, 1600, 6400), (4001, 772, 1088),                            # 128x128
    (6000, 768, 3072),                                                # 192x96
    (1, 36, 128), (17, 100, 192), (33, 772, 1088), (64, 4800, 1600),  # 64 rows or fewer,
    (64, 36, 64), (32, 16388, 128), (33, 16388, 128),                 # with the skinny kernel's side
]


def gemm(gpu, a, w, b, epi, out, bias_dtype=None):
    m, k = a.shape
    n = w.shape[0]
    b = b.to(bias_dtype or a.dtype)
    _lib.check(_lib.load().cgpt_gemm(
        a.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(), m, n, k, a.stride(0), w.stride(0),
        out.stride(0), CODE[a.dtype], CODE[b.dtype], CODE[out.dtype], epi, _lib.TILE_AUTO,
        torch.cuda.current_stream(gpu).cuda_stream), "gemm")
    return out


def problem(gpu, m, n, k, dtype):
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    a = torch.randn(m, k, device=gpu, generator=g).to(dtype)
    w = (torch.randn(n, k, device=gpu, generator=g) * 0.05).to(dtype)
    b = torch.randn(n, device=gpu, generator=g).to(dtype)
    return a, w, b, a.double() @ w.double().t() + b.double()


@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_kgroup_shapes(gpu, m, n, k, dtype):
    a, w, b, ref = problem(gpu, m, n, k, dtype)
    # fp32 sums of K products of |a w| ~ 0.05, as for the other tiles
    tol = 1e-4 * math.sqrt(k / 64)
    out = torch.full((m, n + 4), 7.0, dtype=F32, device=gpu)
    gemm(gpu, a, w, b, _lib.EPI_BIAS, out[:, :n], F32 if m % 2 else None)
    assert (out[:, :n].double() - ref).abs().max() <= tol + 1e-5 * ref.abs().max()
    assert (out[:, n:] == 7.0).all()  # padding of the rows untouched
    x = torch.randn(m, n, device=gpu) * 4
    out = gemm(gpu, a, w, b, _lib.EPI_BIAS_RESID, x.clone())
    assert (out.double() - ref - x.double()).abs().max() <= 2 * tol
    half = gemm(gpu, a, w, b, _lib.EPI_BIAS_GELU, torch.empty(m, n, dtype=dtype, device=gpu))
    want = torch.nn.functional.gelu(ref, approximate="tanh")
    eps = 2.0 ** -8 if dtype == BF16 else 2.0 ** -11
    assert ((half.double() - want).abs() <= eps * want.abs() + tol + 1e-4).all()
    half = x.to(dtype)
    want = ref + half.double()
    gemm(gpu, a, w, b, _lib.EPI_BIAS_RESID, half)
    assert ((half.double() - want).abs() <= eps * want.abs() + 2 * tol).all()


def test_kgroup_repeats_bit_for_bit(gpu):
    a, w, b, _ = problem(gpu, 97, 768, 3072, BF16)
    outs = [gemm(gpu, a, w, b, _lib.EPI_BIAS, torch.empty(97, 768, device=gpu)) for _ in range(3)]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("epi", [_lib.EPI_NONE, _lib.EPI_BIAS, _lib.EPI_BIAS_GELU])
@pytest.mark.parametrize("out_dtype", [BF16, F32])
@pytest.mark.parametrize("m,n,k,pad", [
    (1000, 16388, 128, 0), (1000, 16388, 128, 3),  # one round of 256x256 tiles and 4 columns
    (1000, 16391, 128, 0),                         # ... and 7, rows of odd length
    (300, 33000, 192, 8),                          # two tile rows, 232 columns left
    (1000, 16384, 128, 0),                         # whole rounds: one launch
])
def test_wide_n_whole_rounds(gpu, m, n, k, pad, out_dtype, epi):
    """Wide N whose last columns go to a second launch: both parts, and nothing
    past them."""
    a, w, b, ref = problem(gpu, m, n, k, BF16)
    if epi == _lib.EPI_NONE:
        ref = ref - b.double()
    elif epi == _lib.EPI_BIAS_GELU:
        ref = torch.nn.functional.gelu(ref, approximate="tanh")
    out = torch.full((m, n + pad), 7.0, dtype=out_dtype, device=gpu)
    gemm(gpu, a, w, b, epi, out[:, :n], F32 if pad else None)
    # as above; a bf16 output adds its rounding
    tol = 1e-4 * math.sqrt(k / 64) + (1e-5 if out_dtype is F32 else 2.0 ** -8) * ref.abs().max()
    assert (out[:, :n].double() - ref).abs().max() <= tol
    assert (out[:, n:] == 7.0).all()


@pytest.mark.parametrize("dtype", [BF16, F16, F32])
@pytest.mark.parametrize("row,width", [(0, 772), (2, 772), (0, 769), (1, 769)])
def test_one_row_view(gpu, row, width, dtype):
    """A one-row view counts as contiguous whatever its row stride: neither that
    stride nor its alignment reaches the kernels."""
    from cutilegpt_amd.kernels import cutile_linear_bias

    a, w, b, ref = problem(gpu, 3, 100, 768, dtype)
    wide = torch.zeros(3, width, dtype=dtype, device=gpu)
    wide[:, :768] = a
    out = cutile_linear_bias(wide[row:row + 1, :768], w, b)
    # bit for bit the same kernel's result as for rows of their own
    assert torch.equal(out, cutile_linear_bias(a[row:row + 1].clone(), w, b))
    # 16 bits: one rounding of the output; fp32: sqrt(768) roundings of the running sum
    tol = {F32: 2.0 ** -18, F16: 2.0 ** -10, BF16: 2.0 ** -7}[dtype]
    assert (out.double() - ref[row:row + 1]).abs().max() <= tol * ref.abs().max()


# On either side of the skinny kernel's small weights (12288 of them, 16 rows).
@pytest.mark.parametrize("m,n,k", [(1, 96, 128), (1, 100, 128), (16, 64, 192), (16, 68, 192), (17, 64, 192),
                                   (8, 4, 3072), (8, 8, 3072)])
def test_few_small_weights(gpu, m, n, k):
    test_kgroup_shapes(gpu, m, n, k, BF16)
