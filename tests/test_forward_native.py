"""cgpt_forward: the prefill forward as one native call."""

import ctypes

import pytest
import torch

from cutilegpt_amd import CutileGPT, GPTConfig, _lib

BF16, F32 = torch.bfloat16, torch.float32


@pytest.mark.parametrize("B,T", [(0, 5), (3, 0), (0, 0)])
def test_no_rows_is_a_no_op(B, T):
    """As every launch that it makes: no rows, nothing to do."""
    lib = _lib.load()
    D, H, V = 128, 4, 64
    a = [B, T, D, H, V, 1, 16, _lib.CGPT_F32] + [0] * 12 + [D, V, 0, V, _lib.CGPT_F32, -1, 0] + [0] * 7 + [-1] * 4
    layer = [0] * 12 + [D, D, D, 4 * D, 0, 0]
    rc = lib.cgpt_forward((ctypes.c_int64 * len(a))(*a), (ctypes.c_int64 * len(layer))(*layer), 1.0, 1e-5, None)
    assert rc == 0
    a[26] = 1  # each sequence's last position only
    rc = lib.cgpt_forward((ctypes.c_int64 * len(a))(*a), (ctypes.c_int64 * len(layer))(*layer), 1.0, 1e-5, None)
    assert rc == (0 if T > 0 else -1)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("B,T", [(0, 5), (3, 0), (0, 0)])
def test_empty_batch(gpu, dtype, B, T):
    cfg = GPTConfig(vocab_size=97, block_size=16, n_layer=2, n_head=2, n_embd=64)
    m = CutileGPT(cfg, dtype=dtype, seed=1)
    logits, loss = m(torch.zeros(B, T, dtype=torch.int64, device=gpu))
    assert logits.shape == (B, T, 97) and loss is None
    assert m(torch.zeros(1, 3, dtype=torch.int64, device=gpu))[0].isfinite().all()
