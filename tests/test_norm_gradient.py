"""The final norm carries gradients, as the array op that it replaces did (CPU tensors take that op; the kernel's own cases
are GPU tests)."""
import pytest
import torch

from mxfp4_int8_m5_amd import sc_kernels as S


def test_gradients_of_the_norm():
    g = torch.Generator().manual_seed(0)
    x, w = torch.randn(4, 64, generator=g).to(torch.bfloat16), torch.rand(64, generator=g).to(torch.bfloat16)
    ref = S.rms_norm(x, w, 1e-6)
    assert torch.equal(S.rmsnorm(x, w, 1e-6), ref)
    xg, wg = x.clone().requires_grad_(), w.clone().requires_grad_()
    S.rmsnorm(xg, wg, 1e-6).float().sum().backward()
    n = x.double() * torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + 1e-6)
    # the sum of four bf16 products, each operand rounded once
    torch.testing.assert_close(wg.grad.double(), n.sum(0), rtol=2 ** -6, atol=4 * 2 ** -8 * float(n.abs().max()))
    assert xg.grad.shape == x.shape and xg.grad.abs().max() > 0


@pytest.mark.gpu
def test_model_of_parameters():
    """A model built from parameters that require grad: the same hidden states, a gradient for the final norm's weight."""
    from tests.test_gpu_model import make_tiny
    Q, args, state, packed = make_tiny(4, 2, 64)
    ids = torch.arange(40).cuda()
    params = {k: torch.nn.Parameter(v) for k, v in state.items()}
    h = Q.FusedQwen3(args, params, packed).hidden(ids)
    h.float().sum().backward()
    assert params["model.norm.weight"].grad.abs().max() > 0
    want = Q.FusedQwen3(args, state, packed).hidden(ids)
    # bf16 results of one formula, 1 / sqrt and rsqrt apart: at most two roundings of each value differ
    assert torch.all((h.detach() - want).abs().float() <= 2.0 ** -6 * want.abs().float())
