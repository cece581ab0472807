"""The weighted combine of many rows (a wave each) gives the bits of few rows at a time (a workgroup each): one slot, an odd
count, more than eight, a shared expert's score apart, rows of padding, the shortest and longest row, a ragged last workgroup."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,topk,M,Mp,split", [(512, 1, 1025, 1025, False), (2048, 8, 1100, 1152, False), (2048, 9, 1030, 1056, True),
                                               (1024, 3, 1024, 1026, False), (1536, 17, 1024, 1024, False)])
def test_moe_combine_many_rows(K, topk, M, Mp, split):
    from mxfp4_int8_m5_amd import sc_moe
    g = torch.Generator(device="cuda").manual_seed(K + topk)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(torch.bfloat16)   # noqa: E731
    y, res, w = rnd(M * topk, K), rnd(Mp, K), rnd(K)
    pos = torch.randperm(M * topk, device="cuda", generator=g).to(torch.int32)
    sc = torch.rand(M, topk, device="cuda", generator=g).to(torch.bfloat16)
    few = 500

    def combine(lo, hi):
        m = max(0, min(hi, M) - lo)
        p, s, r = pos[lo * topk:(lo + m) * topk].clone(), sc[lo:lo + m], res[lo:hi].clone()
        if split:
            return sc_moe.moe_combine_split(y, p, s[:, :-1].contiguous(), s[:, -1].contiguous(), r, w, 1e-6, m)[:1]
        return sc_moe.moe_combine(y, p, s.contiguous(), r, w, 1e-6, m)

    parts = [combine(lo, min(Mp, lo + few)) for lo in range(0, Mp, few)]
    for i, got in enumerate(combine(0, Mp)):
        assert torch.equal(got, torch.cat([p[i] for p in parts]))
