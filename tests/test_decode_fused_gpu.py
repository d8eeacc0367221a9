"""cgpt_gemm_partials_ln / cgpt_gemm_partials_gelu: the decode GEMMs that make
their own operand from the previous GEMM's partial products, against the two
launches they replace (same arithmetic, the same bf16 operand up to the order of
a row's sums) and against float64."""

import ctypes

import pytest
import torch

from cutilegpt_amd import CutileGPT, GPTConfig, _lib
from cutilegpt_amd.decode import DecodeSession

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32


def stream(gpu):
    return torch.cuda.current_stream(gpu).cuda_stream


def make(gpu, seed, M, N, K, n_in):
    g = torch.Generator(device=gpu).manual_seed(seed)
    r = lambda *s, scale=1.0: torch.randn(*s, device=gpu, generator=g) * scale
    return dict(parts=r(n_in, M, K), bias=r(K, scale=0.1).to(BF16), x=r(M, K),
                gamma=(1 + r(K, scale=0.1)).to(BF16), beta=r(K, scale=0.1).to(BF16),
                w=r(N, K, scale=0.05).to(BF16))


def plan(M, N, K):
    ns = ctypes.c_int64()
    _lib.check(_lib.load().cgpt_gemm_partials_plan(M, N, K, _lib.CGPT_BF16, ctypes.byref(ns)), "plan")
    return ns.value


# K at the ends of a LayerNorm row, chunks that do not divide K, N with a ragged
# last n-tile and column group, one to sixteen partials.
@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("N,K,n_in", [(4, 64, 1), (132, 128, 3), (768, 768, 12), (2304, 768, 16),
                                      (4800, 1600, 8), (1000, 1984, 9), (512, 2048, 16)])
def test_layernorm_gemm(gpu, M, N, K, n_in):
    lib = _lib.load()
    if not lib.cgpt_decode_fused_ok(M, N, K, K, n_in, 1):
        pytest.skip("not a fused product")
    t = make(gpu, N + K + n_in, M, N, K, n_in)
    ns = plan(M, N, K)
    out, x2 = torch.empty(ns, M, N, device=gpu), torch.empty(M, K, device=gpu)
    _lib.check(lib.cgpt_gemm_partials_ln(
        t["x"].data_ptr(), t["parts"].data_ptr(), n_in, M * K, K, t["bias"].data_ptr(), x2.data_ptr(),
        t["gamma"].data_ptr(), t["beta"].data_ptr(), 1e-5, t["w"].data_ptr(), out.data_ptr(), M, N, K,
        K, N, ns, stream(gpu)), "ln")
    s = t["x"].double() + t["parts"].double().sum(0) + t["bias"].double()
    assert (x2.double() - s).abs().max() <= 1e-5
    h = torch.nn.functional.layer_norm(s, (K,), t["gamma"].double(), t["beta"].double(), 1e-5).to(BF16)
    ref = h.double() @ t["w"].double().t()
    # One bf16 ulp of an operand value here and there, fp32 sums.
    assert ((out.sum(0).double() - ref).norm() / ref.norm()) <= 1e-3


# Up to 1024 columns a wave of either kernel sums the same 256 of a row, in the
# same order, so the operand is the same bit for bit.
@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("N,K,n_in", [(4, 64, 1), (132, 128, 3), (768, 768, 12), (3072, 1024, 16)])
def test_layernorm_gemm_equals_two_launches(gpu, M, N, K, n_in):
    lib = _lib.load()
    assert lib.cgpt_decode_fused_ok(M, N, K, K, n_in, 1)
    t = make(gpu, N + K + n_in, M, N, K, n_in)
    ns = plan(M, N, K)
    out, two = torch.empty(ns, M, N, device=gpu), torch.empty(ns, M, N, device=gpu)
    x2, x3, h = torch.empty(M, K, device=gpu), torch.empty(M, K, device=gpu), torch.empty(M, K, dtype=BF16, device=gpu)
    _lib.check(lib.cgpt_gemm_partials_ln(
        t["x"].data_ptr(), t["parts"].data_ptr(), n_in, M * K, K, t["bias"].data_ptr(), x2.data_ptr(),
        t["gamma"].data_ptr(), t["beta"].data_ptr(), 1e-5, t["w"].data_ptr(), out.data_ptr(), M, N, K,
        K, N, ns, stream(gpu)), "ln")
    _lib.check(lib.cgpt_add_layernorm_partials(
        t["x"].data_ptr(), t["parts"].data_ptr(), n_in, M * K, K, t["bias"].data_ptr(), x3.data_ptr(),
        t["gamma"].data_ptr(), t["beta"].data_ptr(), h.data_ptr(), M, K, 1e-5, _lib.CGPT_F32, _lib.CGPT_F32,
        _lib.CGPT_BF16, _lib.CGPT_BF16, stream(gpu)), "add_ln")
    _lib.check(lib.cgpt_gemm_partials(h.data_ptr(), t["w"].data_ptr(), two.data_ptr(), M, N, K, K, K, N,
                                      ns, _lib.CGPT_BF16, stream(gpu)), "partials")
    assert torch.equal(x2, x3) and torch.equal(out, two)


@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("N,K,n_in", [(4, 64, 1), (132, 192, 3), (768, 3072, 5), (1600, 2560, 16),
                                      (512, 2048, 9)])
def test_gelu_gemm(gpu, M, N, K, n_in):
    lib = _lib.load()
    if not lib.cgpt_decode_fused_ok(M, N, K, K, n_in, 0):
        pytest.skip("not a fused product")
    t = make(gpu, N + K + n_in, M, N, K, n_in)
    ns = plan(M, N, K)
    out = torch.empty(ns, M, N, device=gpu)
    _lib.check(lib.cgpt_gemm_partials_gelu(
        t["parts"].data_ptr(), n_in, M * K, K, t["bias"].data_ptr(), t["w"].data_ptr(), out.data_ptr(),
        M, N, K, K, N, ns, stream(gpu)), "gelu")
    f = torch.empty(M, K, dtype=BF16, device=gpu)
    _lib.check(lib.cgpt_partials_bias_act(t["parts"].data_ptr(), n_in, M * K, K, t["bias"].data_ptr(),
                                          _lib.CGPT_BF16, f.data_ptr(), K, M, K, _lib.EPI_BIAS_GELU,
                                          _lib.CGPT_BF16, stream(gpu)), "act")
    two = torch.empty(ns, M, N, device=gpu)
    _lib.check(lib.cgpt_gemm_partials(f.data_ptr(), t["w"].data_ptr(), two.data_ptr(), M, N, K, K, K, N,
                                      ns, _lib.CGPT_BF16, stream(gpu)), "partials")
    assert torch.equal(out, two)  # the same operand, sums and order


def test_fused_refuses(gpu):
    lib = _lib.load()
    assert lib.cgpt_decode_fused_ok(3, 768, 768, 768, 4, 1) == 0   # rows
    assert lib.cgpt_decode_fused_ok(1, 768, 800, 800, 4, 1) == 0   # K % 64
    assert lib.cgpt_decode_fused_ok(1, 768, 2112, 2112, 4, 1) == 0  # LayerNorm row
    assert lib.cgpt_decode_fused_ok(1, 768, 768, 768, 17, 1) == 0  # partials
    t = make(gpu, 1, 1, 64, 64, 2)
    out = torch.empty(1, 1, 64, device=gpu)
    args = [t["x"].data_ptr(), t["parts"].data_ptr(), 2, 64, 64, t["bias"].data_ptr(), t["x"].data_ptr(),
            t["gamma"].data_ptr(), t["beta"].data_ptr(), 1e-5, t["w"].data_ptr(), out.data_ptr(), 1, 64,
            64, 64, 64, 1, stream(gpu)]
    assert lib.cgpt_gemm_partials_ln(*args) == -1  # x_out is x


@pytest.mark.parametrize("B", [1, 2])
@pytest.mark.parametrize("shape", [(3, 4, 64), (2, 4, 128), (2, 12, 768)])
def test_fused_session_equals_unfused(gpu, B, shape):
    L, H, D = shape
    cfg = GPTConfig(vocab_size=512, block_size=64, n_layer=L, n_head=H, n_embd=D)
    m = CutileGPT(cfg, dtype=BF16, seed=3)
    idx = torch.randint(0, 512, (B, 9), generator=torch.Generator().manual_seed(4)).to(gpu)
    logits = []
    for fused in (True, False):
        s = DecodeSession(m, B, 9, 8)
        assert s.fused
        s.fused = fused
        s.prefill(idx)
        s.step.zero_()
        rows = []
        for i in range(6):
            s.ids.copy_((idx[:, i] * 7 + i) % 512)
            s.step_logits()
            s.step.add_(1)
            rows.append(s.logits.clone())
        logits.append(torch.stack(rows))
    # The two differ by the order of a LayerNorm row's sums, which may flip a
    # bf16 rounding of its output.
    assert (logits[0] - logits[1]).norm() / logits[1].norm() <= 5e-3
