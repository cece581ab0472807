"""RMSNorm, quantization and router linear of one row in one launch: the bits of the separate launches, at every width the kernel is built
for and at the edges of its tiles of router rows; what it does not take is left to those."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [512, 1024, 1536, 2048])
@pytest.mark.parametrize("e,k", [(1, 1), (7, 7), (16, 2), (17, 4), (33, 8), (63, 8), (64, 64), (257, 8)])
def test_equals_the_separate_launches(d, e, k):
    from mxfp4_int8_m5_amd import sc_kernels as S, sc_moe as M
    g = torch.Generator(device="cuda").manual_seed(d + e)
    w, gate = ((torch.randn(s, device="cuda", generator=g) * 0.05 + o).bfloat16() for s, o in ((d, 1), ((e, d), 0)))
    for scale in (1.0, 1e-6, 1e4, 0.0):
        for renorm in (True, False):
            x = (torch.randn(1, d, device="cuda", generator=g) * scale).bfloat16()
            xq, xs, xn = S.rmsnorm_quant_n(x, w, 1e-5, 1)
            want = (xq, xs, xn, *M.route(S.linear_bf16(xn, gate), k, renorm))
            got = M.norm_route(x, w, 1e-5, gate, k, renorm)
            for a, b in zip(got, want):
                assert a.dtype == b.dtype and a.shape == b.shape
                assert torch.equal(a.view(torch.int16) if a.dtype == torch.bfloat16 else a, b.view(torch.int16) if b.dtype == torch.bfloat16 else b)


def test_left_to_the_separate_launches():
    from mxfp4_int8_m5_amd import sc_moe as M
    t = lambda *s: torch.ones(s, device="cuda", dtype=torch.bfloat16)   # noqa: E731
    assert M.norm_route(t(1, 2560), t(2560), 1e-5, t(8, 2560), 2) is None
    assert M.norm_route(t(1, 576), t(576), 1e-5, t(8, 576), 2) is None
    assert M.norm_route(t(2, 512), t(512), 1e-5, t(8, 512), 2) is None
    assert M.norm_route(t(1, 512), t(512), 1e-5, t(8, 512).float(), 2) is None
    assert M.norm_route(t(1, 512), t(512), 1e-5, t(8, 512).requires_grad_(), 2) is None
    assert M.norm_route(t(513)[1:].view(1, 512), t(512), 1e-5, t(8, 512), 2) is None
    assert M.norm_route(t(1, 512), t(512), 1e-5, t(8, 512), 2) is not None
