"""Decode attention with two query heads of a KV head to a workgroup: both sides of the row count it starts at (3072) and of the one-workgroup
limit, head groups of even and odd sizes, ranges that are and are not paired, against float64; the fused form against the two calls."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("hq,hk", [(4, 2), (6, 2), (4, 1), (3, 3)])
@pytest.mark.parametrize("n", [1, 128, 129, 3071, 3072, 3073, 3900])
def test_against_float64_and_fused(n, hq, hk, d):
    from mxfp4_int8_m5_amd import sc_kernels as S
    g = torch.Generator(device="cuda").manual_seed(n + d + hq)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g).bfloat16()   # noqa: E731
    k, v = rnd(hk, 4000, d), rnd(hk, 4000, d)
    y, qn, kn = rnd(1, (hq + 2 * hk) * d), rnd(d), rnd(d)
    freq = 1e4 ** (-torch.arange(d // 2, device="cuda", dtype=torch.float32) / (d // 2))
    for splits in (None, 31, 32, 33, 64):
        k1, v1, k2, v2 = k.clone(), v.clone(), k.clone(), v.clone()
        q = S.qkv_headnorm_rope(y, qn, kn, 1e-6, 1, hq, hk, d, k1, v1, n - 1, freq)
        for pos in (n, torch.tensor([n - 1], device="cuda")):
            got = S.attn_decode(q, k1, v1, pos, splits=splits)
            p = torch.softmax(torch.einsum("hd,hnd->hn", q[:, 0].double(), k1[:, :n].double().repeat_interleave(hq // hk, 0)) * d ** -0.5, -1)
            want = torch.einsum("hn,hnd->hd", p, v1[:, :n].double().repeat_interleave(hq // hk, 0))
            # float32 sums and weights (exponents to 2^-21 of scores up to some tens), one rounding to bf16
            assert float((got.double().reshape(hq, d) - want).norm() / want.norm()) < 2 ** -8
            fused = S.attn_decode_qkv(y, qn, kn, 1e-6, hq, hk, d, k2, v2, pos if torch.is_tensor(pos) else n - 1, freq, splits=splits)
            assert torch.equal(fused.view(torch.int16), got.view(torch.int16)) and torch.equal(k1, k2) and torch.equal(v1, v2)


@pytest.mark.parametrize("pos", [-1, 4000])
def test_a_position_outside_the_cache_gives_zeros(pos):
    from mxfp4_int8_m5_amd import sc_kernels as S
    k, v, q = (torch.randn(s, device="cuda").bfloat16() for s in ((2, 4000, 128), (2, 4000, 128), (4, 128)))
    assert not S.attn_decode(q, k, v, torch.tensor([pos], device="cuda")).any()
