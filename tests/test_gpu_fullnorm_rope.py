"""The fused q/k norm + rotary embedding + cache append of the full-width norm, and the plain RMSNorm rows, where their
kernels change: widths held by a wave and widths that are not, head dims with and without a lane-aligned rotation partner."""
import numpy as np
import pytest
import torch

from oracle import bf16, linear
from tests.util import dev, host, llm_acts

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    from mxfp4_int8_m5_amd import sc_kernels
    return sc_kernels


@pytest.mark.parametrize("h,d", [(16, 128), (32, 64), (2, 256), (4, 512), (32, 16), (2, 128), (12, 96), (3, 4)])
@pytest.mark.parametrize("L,pos,on_device", [(1, 0, False), (1, 37, True), (7, 5, False)])
def test_fullnorm_rope(S, h, d, L, pos, on_device):
    rng = np.random.default_rng(h * d + L)
    W, rows = h * d, 48
    y = llm_acts(rng, L, 3 * W)[0]
    qn, kn = llm_acts(rng, 1, W)[0][0], llm_acts(rng, 1, W)[0][0]
    kc = torch.zeros((h, rows, d), dtype=torch.bfloat16, device="cuda")
    vc = torch.zeros_like(kc)
    inv = (1.0 / (1e4 ** (torch.arange(d // 2).float() / (d // 2)))).cuda()
    q = S.qkv_fullnorm_rope(dev(y), dev(qn), dev(kn), 1e-5, L, h, d, kc, vc,
                            torch.tensor([pos], device="cuda") if on_device else pos, inv)
    ang = (torch.arange(pos, pos + L).float()[:, None] * inv.cpu()[None]).double()
    for got, bits, turn in zip((q, kc[:, pos:pos + L], vc[:, pos:pos + L]), linear.fullnorm(y, qn, kn, 1e-5, L, h, d),
                               (True, True, False)):
        x = torch.from_numpy(bf16.from_bits(bits).astype(np.float64)).reshape(h, L, d)
        if turn:
            a, b = x[..., :d // 2], x[..., d // 2:]
            x = torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1)
        g = got.double().cpu()
        # one rounding to bf16 (8-bit significand: at most half a unit in the last place, 2^-8 of the value) and float32
        # arithmetic on operands up to the largest value (a few times 2^-24 of it, the float32 sine and cosine included)
        assert ((g - x).abs() <= x.abs() * 2.0 ** -8 + 1e-6 * x.abs().amax()).all()
    keep = torch.ones(rows, dtype=torch.bool)
    keep[pos:pos + L] = False
    assert not kc[:, keep].any() and not vc[:, keep].any()
    with pytest.raises(ValueError):
        S.qkv_fullnorm_rope(dev(y), dev(qn), dev(kn), 1e-5, L, h, d, kc, vc, rows - L + 1, inv)


@pytest.mark.parametrize("m,k", [(1, 512), (5, 2048), (9, 4096), (3, 640), (2, 8192), (4, 4)])
def test_rmsnorm_rows(S, m, k):
    rng = np.random.default_rng(m * k)
    x, w = llm_acts(rng, m, k)[0], llm_acts(rng, 1, k)[0][0]
    assert np.array_equal(host(S.rmsnorm(dev(x), dev(w), 1e-6)), linear.rmsnorm(x, w, 1e-6))


def test_rmsnorm_array_op(S, monkeypatch):
    """Callers that differentiate or transform the norm, and tensors off the current device, get the array op."""
    from mxfp4_int8_m5_amd.fused_qwen3 import rms_norm
    x, w = torch.randn(5, 256, device="cuda").to(torch.bfloat16), torch.rand(256, device="cuda").to(torch.bfloat16)
    ref = rms_norm(x, w, 1e-6)
    for t in (x, w):
        g = t.clone().requires_grad_()
        a = (g, w) if t is x else (x, g)
        S.rmsnorm(*a, 1e-6).float().sum().backward()
        want = t.clone().requires_grad_()
        rms_norm(*((want, w) if t is x else (x, want)), 1e-6).float().sum().backward()
        assert torch.equal(g.grad, want.grad)
        with torch.no_grad():
            assert not S.rmsnorm(*a, 1e-6).requires_grad
    assert torch.equal(torch.func.vmap(lambda r: S.rmsnorm(r[None], w, 1e-6)[0])(x), ref)
    assert S.rmsnorm(x[:0], w, 1e-6).shape == (0, 256)
    assert torch.equal(S.rmsnorm(x.t().contiguous().t(), w, 1e-6), ref)          # columns first
    odd = torch.randn(3, 250, device="cuda").to(torch.bfloat16)
    assert torch.equal(S.rmsnorm(odd, w[:250], 1e-6), rms_norm(odd, w[:250], 1e-6))
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: x.device.index + 1)
    monkeypatch.setattr(S._lib, "native", lambda: pytest.fail("launched on the current device"))
    assert torch.equal(S.rmsnorm(x, w, 1e-6), ref)


@pytest.mark.parametrize("h,d", [(1, 516), (2, 1024), (1, 16384)])
@pytest.mark.parametrize("L,pos,on_device", [(1, 37, True), (7, 5, False)])
def test_fullnorm_rope_long_heads(S, h, d, L, pos, on_device):
    test_fullnorm_rope(S, h, d, L, pos, on_device)
