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


# every form of the kernel: one to four turns of a row, each full and not; several batches of three and of four, full and not,
# with one tile and with several per workgroup (the next tile's first batch is requested behind this one's last)
@pytest.mark.parametrize("m,n,k", [(3, 33, 576), (16, 40, 1024), (5, 16, 1088), (16, 9001, 1536), (4, 20, 1984), (1, 17000, 2112),
                                   (2, 17000, 2560), (1, 9001, 4096), (2, 8200, 4608), (2, 9001, 3584), (16, 50, 6400), (1, 3, 8192)])
def test_linear_bf16_forms(S, m, n, k):
    test_linear_bf16_kernel(S, m, n, k)


def test_linear_bf16_kernel(S, m=2, n=300, k=2048):
    """The kernel itself, whichever op linear_bf16 chooses for the shape; nothing outside the rows reaches the sums."""
    g = torch.Generator(device="cuda").manual_seed(m * n + k)
    x, w = (torch.full((r * k + 128,), float("nan"), device="cuda", dtype=torch.bfloat16) for r in (m, n))
    x, w = x[64:-64].view(m, k), w[64:-64].view(n, k)
    x.copy_(torch.randn(m, k, device="cuda", generator=g)), w.copy_(torch.randn(n, k, device="cuda", generator=g))
    y = torch.empty(m, n, device="cuda", dtype=torch.bfloat16)
    S._lib.native().scmx_linear_bf16(x, w, y, m, n, k)
    xd, wd = x.double(), w.double()
    ref, mag = xd @ wd.T, xd.abs() @ wd.abs().T
    assert ((y.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + mag * k * 2.0 ** -24).all()
