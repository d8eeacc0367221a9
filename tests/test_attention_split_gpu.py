"""fp32 attention of head_dim 64 on split bf16 operands (csrc/attention_split.hip)
against float64: edges of the 16-query, 64-key and 64/128-query tiles, and inputs
that bf16 parts cannot hold."""

import math

import pytest
import torch

from cutilegpt_amd import cutile_causal_attention

pytestmark = pytest.mark.gpu


def randn(gpu, *shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(gpu)


def exact(q, k, v):
    q, k, v = (t.double() for t in (q, k, v))
    T = q.shape[2]
    s = (q @ k.transpose(2, 3).contiguous()) / math.sqrt(q.shape[3])
    s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1), -math.inf)
    return torch.softmax(s, -1) @ v


# fp32's own error: 2^-24 of each score (|s| up to ~6 in base 2), of each of the
# T probabilities and of the sums; 32 roundings cover them at |v| <= 5.
TOL = 32 * 5 * 2.0 ** -24


@pytest.mark.parametrize("B,H,T", [(1, 1, 1), (1, 2, 15), (2, 3, 17), (1, 3, 63), (1, 3, 64), (1, 3, 65),
                                   (3, 5, 129), (1, 12, 200), (32, 32, 130), (128, 8, 129)])
def test_split_attention_shapes(gpu, B, H, T):
    q, k, v = (randn(gpu, B, H, T, 64, seed=i) for i in range(3))
    out = cutile_causal_attention(q, k, v, H)
    assert (out.double() - exact(q, k, v)).abs().max() <= TOL


def test_split_attention_strided_views(gpu):
    B, H, T = 2, 4, 70
    x = randn(gpu, B, T, 3, H, 64)
    q, k, v = (x[:, :, i].transpose(1, 2) for i in range(3))
    out = cutile_causal_attention(q, k, v, H)
    assert (out.double() - exact(q, k, v)).abs().max() <= TOL


def test_split_attention_non_finite(gpu):
    B, H, T = 1, 2, 200
    q, k, v = (randn(gpu, B, H, T, 64, seed=i) for i in range(3))
    q[..., 0] = -q[..., 0].abs() - 0.1
    k[0, 0, 37, 0] = math.inf       # score -inf for every query: weight 0
    v[0, 1, 80, 5] = math.inf       # column 5 of later queries
    v[0, 1, 150, 9] = math.nan
    k[0, 0, 3, 1] = 3.4e38          # infinite in bf16 only; the scores stay finite
    q[0, 0, :, 1] = 1e-39
    out = cutile_causal_attention(q, k, v, H)
    kk = k.double()
    kk[0, 0, 37, 0] = 1e300         # float64's stand-in: weight exactly 0
    ref = exact(q, kk, v.nan_to_num(0, 0, 0))
    assert (out[0, 0].double() - ref[0, 0]).abs().max() <= TOL
    # Queries before the 16-key tile of the odd value do not see it; those at or
    # after its key do.
    assert (out[0, 1, :80].double() - ref[0, 1, :80]).abs().max() <= TOL
    assert torch.isinf(out[0, 1, 80:144, 5]).all() and (out[0, 1, 80:, 5] > 0).all()
    assert torch.isnan(out[0, 1, 150:, 9]).all()
    cols = [c for c in range(64) if c not in (5, 9)]
    assert (out[0, 1][:, cols].double() - ref[0, 1][:, cols]).abs().max() <= TOL


@pytest.mark.parametrize("scale", [1e-28, 1e-30, 1e-36])
def test_split_attention_tiny_values(gpu, scale):
    B, H, T = 1, 2, 100
    q, k, v = (randn(gpu, B, H, T, 64, seed=i) for i in range(3))
    v[..., 7:20] *= scale
    out, ref = cutile_causal_attention(q, k, v, H).double(), exact(q, k, v)
    col = (out - ref).norm(dim=2) / ref.norm(dim=2)
    assert col.max() <= TOL, col.max()


def row_err(out, ref):
    """Largest error of a row over the row's norm."""
    return ((out.double() - ref).norm(dim=-1) / ref.norm(dim=-1)).max()


# Elements of Q and K of inverse scales: in every column, or in every second one
# (an ordinary value beside each small one).  Ordinary scores, so TOL holds.
@pytest.mark.parametrize("step", [1, 2])
@pytest.mark.parametrize("e", [-125, -123, -100, -90, -70, 70, 90, 100, 115, 123, 125])
def test_split_attention_inverse_scales(gpu, e, step):
    q, k, v = (randn(gpu, 1, 2, 150, 64, seed=i) for i in range(3))
    q[..., ::step] *= 2.0 ** e
    k[..., ::step] *= 2.0 ** -e
    out = cutile_causal_attention(q, k, v, 2)
    assert (out.double() - exact(q, k, v)).abs().max() <= TOL


# Early rows see small values of V alone; the same columns are ordinary for
# later keys.  Relative to each row: the bound for |v| <= 5 over a row's norm of
# about 8 / sqrt(150).
@pytest.mark.parametrize("e", [100, 115, 120, 125])
def test_split_attention_tiny_values_before_others(gpu, e):
    q, k, v = (randn(gpu, 1, 2, 150, 64, seed=i) for i in range(3))
    v[:, :, :70] *= 2.0 ** -e
    out, ref = cutile_causal_attention(q, k, v, 2), exact(q, k, v)
    assert row_err(out[:, :, :70], ref[:, :, :70]) <= TOL
    assert row_err(out[:, :, 70:], ref[:, :, 70:]) <= TOL


# Small probabilities beside large ones whose values are zero: the result is the
# small ones' alone.  fp32 rounds the exponent of 2^-g to 2^-17 absolute (2^-18
# in the score, 2^-18 in its scaling), 8 such errors of 0.7 * 2^-17 each.
@pytest.mark.parametrize("g", [60, 100, 115, 120, 124])
def test_split_attention_tiny_probabilities(gpu, g):
    q, k, v = (randn(gpu, 1, 1, 100, 64, seed=i) for i in range(3))
    q[..., 0], k[..., 0] = 1.0, 0.0
    q[..., 1:] *= 1e-3
    k[..., ::2, 0] = -g * math.log(2.0) * 8   # every second key: 2^-g of the others
    v[..., ::2, :] *= 2.0 ** 100
    v[..., 1::2, :] = 0.0
    out, ref = cutile_causal_attention(q, k, v, 1), exact(q, k, v)
    assert row_err(out[:, :, 1:], ref[:, :, 1:]) <= 8 * 2.0 ** -17
