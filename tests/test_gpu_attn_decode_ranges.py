"""Decode attention over its row ranges against float64: contexts around the one-workgroup limit (128 rows), the first split length, counts
that leave ranges short or empty, and more ranges than the merge takes at once."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("n", [1, 15, 16, 127, 128, 129, 145, 500, 512, 513, 1040, 2999])
@pytest.mark.parametrize("splits", [None, 1, 3, 16, 17, 33, 64])
def test_against_float64(n, d, splits):
    from mxfp4_int8_m5_amd import sc_kernels as S
    g = torch.Generator(device="cuda").manual_seed(n + d)
    k, v, q = (torch.randn(s, device="cuda", generator=g).bfloat16() for s in ((2, 3000, d), (2, 3000, d), (4, d)))
    p = torch.softmax(torch.einsum("hd,hnd->hn", q.double(), k[:, :n].double().repeat_interleave(2, 0)) * d ** -0.5, -1)
    want = torch.einsum("hn,hnd->hd", p, v[:, :n].double().repeat_interleave(2, 0))
    for pos in (n, torch.tensor([n - 1], device="cuda")):
        got = S.attn_decode(q, k, v, pos, splits=splits).double().reshape(4, d)
        # float32 sums and weights (exponents to 2^-21 of scores up to about 8), one rounding to bf16
        assert float((got - want).norm() / want.norm()) < 2 ** -8
