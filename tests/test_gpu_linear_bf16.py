"""The few-row bf16 linear where its kernel changes: one and sixteen rows, a ragged last tile of outputs, fewer chunks of
64 columns than waves, one more than a batch of loads; and the calls that stay with the array op."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    from mxfp4_int8_m5_amd import sc_kernels
    return sc_kernels


@pytest.mark.parametrize("m,n,k", [(1, 1, 64), (1, 64, 2048), (16, 17, 448), (3, 16, 512), (2, 33, 2112), (2, 1000, 4096), (1, 9000, 1472)])
def test_linear_bf16(S, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m * n + k)
    x, w = (torch.randn(r, k, device="cuda", generator=g).to(torch.bfloat16) for r in (m, n))
    y = S.linear_bf16(x, w)
    ref, mag = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    # one rounding to bf16 and k float32 additions
    assert y.shape == (m, n) and ((y.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + mag * k * 2.0 ** -24).all()


def test_linear_bf16_array_op(S):
    x, w = (torch.randn(r, 256, device="cuda").to(torch.bfloat16) for r in (4, 40))
    ref = x.float() @ w.float().T
    close = lambda y: torch.testing.assert_close(y.float(), ref, rtol=2e-2, atol=2e-2)   # noqa: E731
    close(S.linear_bf16(x.t().contiguous().t(), w))                    # columns first
    close(torch.func.vmap(lambda r: S.linear_bf16(r[None], w)[0])(x))
    xg = x.clone().requires_grad_()
    S.linear_bf16(xg, w).float().sum().backward()
    assert xg.grad.shape == x.shape
    t = torch.randn_like(x)
    _, jt = torch.func.jvp(lambda v: S.linear_bf16(v, w), (x,), (t,))
    torch.testing.assert_close(jt.float(), t.float() @ w.float().T, rtol=2e-2, atol=2e-2)
    assert S.linear_bf16(x[0], w).shape == (40,) and S.linear_bf16(x[:0], w).shape == (0, 40)
    with torch.autocast("cuda", torch.float16):
        assert S.linear_bf16(x, w).dtype == torch.float16
    with pytest.raises(RuntimeError):
        S.linear_bf16(x[:, :64], w)


def test_linear_bf16_off_the_current_device(S, monkeypatch):
    """Kernels are launched on the current device: tensors of another GPU get the array op, which runs on theirs."""
    x, w = (torch.randn(r, 256, device="cuda").to(torch.bfloat16) for r in (4, 40))
    ref = x @ w.T
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: x.device.index + 1)
    monkeypatch.setattr(S._lib, "native", lambda: pytest.fail("launched on the current device"))
    assert torch.equal(S.linear_bf16(x, w), ref)
