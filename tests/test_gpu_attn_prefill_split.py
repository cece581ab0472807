"""Prefill attention with the keys cut into ranges, where that can go wrong: a query tile that ends in the first range beside
one that does not, a range that some queries do not reach, one pair of tiles per range, more ranges than pairs, and head
counts that are whole turns of the XCDs (the heads' order then differs) beside those that are not."""
import pytest
import torch



def test_ranges_stay_in_bounds():
    from mxfp4_int8_m5_amd import sc_kernels as S
    for L in (0, 1, 127, 128, 129, 1000, 5000):
        for off in (0, 1, 200, 4000, 100000):
            for hq in (1, 2, 16, 48, 300):
                s = S.attn_prefill_splits(L, off, hq)
                assert 1 <= s <= 64 and (s == 1 or s * hq * -(-L // 128) <= 256)
    assert [S.attn_prefill_splits(*a) for a in ((1500, 0, 16), (8, 200, 16), (32, 300, 16), (100, 4000, 16), (1000, 1000, 16))] == [1, 1, 3, 16, 2]


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [128 ** -0.5, 0.07, 0.031])
@pytest.mark.parametrize("hq,hk,L,off,splits", [(2, 1, 1, 127, 2), (2, 2, 1, 128, 2), (4, 2, 32, 60, 1), (4, 2, 32, 1000, 8), (2, 1, 129, 1000, 3),
                                                (2, 2, 300, 0, 2), (3, 3, 200, 120, 64), (1, 1, 2, 5000, 13),
                                                (8, 2, 130, 700, 3), (16, 16, 40, 900, 8), (16, 8, 300, 200, 2), (24, 8, 1, 500, 4)])
def test_attn_prefill_split(hq, hk, L, off, splits, scale):
    from mxfp4_int8_m5_amd import sc_kernels as S
    n, d = off + L, 128
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(torch.bfloat16)   # noqa: E731
    q, kc, vc = rnd(L, hq, d), rnd(hk, n + 3, d), rnd(hk, n + 3, d)
    kc[:, n:], vc[:, n:] = float("nan"), float("nan")
    o = S.attn_prefill(q.transpose(0, 1), kc, vc, off, scale, splits).view(L, hq, d).double().cpu()
    k, v = (t[:, :n].double().cpu().repeat_interleave(hq // hk, 0) for t in (kc, vc))
    s = q.transpose(0, 1).double().cpu() @ k.transpose(1, 2).contiguous() * scale
    seen = torch.arange(n) <= off + torch.arange(L)[:, None]
    p = torch.softmax(s.masked_fill(~seen, -torch.inf), -1)
    ref, mag = (p @ v).transpose(0, 1), (p @ v.abs()).transpose(0, 1)
    # a bf16 rounding of each weight and one of the result (2^-8 each); float32 sums and exponents are far below
    assert ((o - ref).abs() <= 2.0 ** -8 * (mag + ref.abs()) * 1.05 + 1e-6).all()
