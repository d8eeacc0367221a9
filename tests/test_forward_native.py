"""cgpt_forward: the prefill forward as one native call."""

import ctypes

import pytest
import torch

from cutilegpt_amd import CutileGPT, GPTConfig, _lib
from cutilegpt_amd.decode import KVCache

BF16, F32 = torch.bfloat16, torch.float32


def call(a, layers, probe=None, n_a=None):
    """(status, tag of the failed launch)"""
    failed = ctypes.c_int(99)
    rc = _lib.load().cgpt_forward(
        (ctypes.c_int64 * len(a))(*a), len(a) if n_a is None else n_a, (ctypes.c_int64 * len(layers))(*layers),
        1.0, 1e-5, None if probe is None else ctypes.cast(probe, ctypes.c_void_p), ctypes.byref(failed), None)
    return rc, failed.value


def empty_args(B, T, n_layer=1):
    D, H, V = 128, 4, 64
    a = [B, T, D, H, V, n_layer, 16, _lib.CGPT_F32] + [0] * 12 + [D, V, 0, V, _lib.CGPT_F32, -1, 0] + [0] * 7
    layer = [0] * 12 + [D, D, D, 4 * D]
    return a + [-1] * 4, layer * n_layer + [0, 0]


@pytest.mark.parametrize("B,T", [(0, 5), (3, 0), (0, 0)])
def test_no_rows_is_a_no_op(B, T):
    """As every launch that it makes: no rows, nothing to do."""
    a, layers = empty_args(B, T)
    assert call(a, layers)[0] == 0
    a[26] = 1  # each sequence's last position only
    assert call(a, layers)[0] == (0 if T > 0 else -1)


def test_probe_failed_and_argument_count():
    a, layers = empty_args(0, 5, n_layer=2)
    seen = []

    def stop_after(n):
        def probe(tag, start):
            seen.append((_lib.FORWARD_TAGS[tag], start))
            return int(len(seen) == n)
        return _lib.FORWARD_PROBE(probe)

    assert call(a, layers, stop_after(0))[0] == 0
    layer = ["gemm_qkv", "attention", "gemm_proj", "ln", "gemm_fc_gelu", "gemm_mlp_proj", "ln"]
    order = ["embedding"] + 2 * layer + ["lm_head"]
    assert seen == [(t, s) for t in order for s in (1, 0)]
    seen.clear()
    assert call(a, layers, stop_after(4)) == (-1, _lib.FORWARD_TAGS.index("gemm_qkv"))
    assert len(seen) == 4
    assert call(a, layers, n_a=37) == (-1, -1)
    a[21] = -1                       # the head's rows
    assert call(a, layers) == (-1, _lib.FORWARD_TAGS.index("lm_head"))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("B,T", [(0, 5), (3, 0), (0, 0)])
def test_empty_batch(gpu, dtype, B, T):
    cfg = GPTConfig(vocab_size=97, block_size=16, n_layer=2, n_head=2, n_embd=64)
    m = CutileGPT(cfg, dtype=dtype, seed=1)
    logits, loss = m(torch.zeros(B, T, dtype=torch.int64, device=gpu))
    assert logits.shape == (B, T, 97) and loss is None
    assert m(torch.zeros(1, 3, dtype=torch.int64, device=gpu))[0].isfinite().all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16])
def test_probed_forward_is_the_forward(gpu, dtype):
    cfg = GPTConfig(vocab_size=97, block_size=64, n_layer=2, n_head=2, n_embd=64)
    m = CutileGPT(cfg, dtype=dtype, seed=1)
    idx = torch.randint(0, 97, (3, 33), generator=torch.Generator().manual_seed(2)).to(gpu)
    marks = []
    probed = m.forward(idx, probe=lambda tag, start: marks.append((tag, start)))[0]
    assert torch.equal(probed, m(idx)[0])
    layer = ["gemm_qkv", "attention", "gemm_proj", "ln", "gemm_fc_gelu", "gemm_mlp_proj", "ln"]
    assert marks == [(t, s) for t in ["embedding"] + 2 * layer + ["lm_head"] for s in (True, False)]

    class Stop(Exception):
        pass

    def probe(tag, start):
        marks.append(tag)
        if tag == "attention":
            raise Stop("here")

    marks.clear()
    with pytest.raises(Stop, match="here"):
        m.forward(idx, probe=probe)
    assert marks == ["embedding", "embedding", "gemm_qkv", "gemm_qkv", "attention"]
    assert torch.equal(m(idx)[0], probed)


@pytest.mark.gpu
def test_error_names_the_launch(gpu):
    cfg = GPTConfig(vocab_size=97, block_size=16, n_layer=2, n_head=2, n_embd=64)
    m = CutileGPT(cfg, dtype=BF16, seed=1)
    cache = KVCache(2, 1, 2, 4, 32, BF16, gpu)  # four rows for five positions
    with pytest.raises(ValueError, match="kv_store"):
        m._forward(torch.zeros(1, 5, dtype=torch.int64, device=gpu), cache=cache)
