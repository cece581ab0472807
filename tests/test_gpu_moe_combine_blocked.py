"""The weighted combine whose codes leave in the blocked layout: the bits of the row form, the shortest and longest row, padding rows;
shapes and row counts that stay by rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,topk,M,Mp,blocked", [(512, 1, 1025, 1056, True), (1024, 3, 1024, 1024, True), (1536, 17, 1030, 1056, True),
                                                 (2048, 8, 1100, 1152, True), (2048, 8, 990, 992, False), (2048, 8, 1030, 1030, False),
                                                 (4096, 2, 1024, 1024, False)])
def test_same_bits_as_by_rows(K, topk, M, Mp, blocked):
    from mxfp4_int8_m5_amd import sc_kernels as S
    from mxfp4_int8_m5_amd import sc_moe
    g = torch.Generator(device="cuda").manual_seed(K + topk)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(torch.bfloat16)   # noqa: E731
    y, res, w = rnd(M * topk, K), rnd(Mp, K), rnd(K)
    pos = torch.randperm(M * topk, device="cuda", generator=g).to(torch.int32)
    sc = torch.rand(M, topk, device="cuda", generator=g).to(torch.bfloat16)
    want = sc_moe.moe_combine(y, pos, sc, res, w, 1e-6, M)
    h, xq, xs = sc_moe.moe_combine(y, pos, sc, res, w, 1e-6, M, blocked=True)
    assert isinstance(xq, S.BlockedXq) == blocked
    assert torch.equal(h, want[0]) and torch.equal(xs, want[2]) and torch.equal(xq.rows() if blocked else xq, want[1])


@pytest.mark.parametrize("K,topk,M,Mp", [(512, 2, 37, 64), (1536, 5, 100, 128), (2048, 9, 70, 96)])
def test_the_shared_expert_apart(K, topk, M, Mp):
    """The C entry with the last slot's scores in a tensor of their own: the bits of the row form."""
    from mxfp4_int8_m5_amd import _lib
    from mxfp4_int8_m5_amd import sc_kernels as S
    g = torch.Generator(device="cuda").manual_seed(K + topk)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(torch.bfloat16)   # noqa: E731
    y, res, w = rnd(M * topk, K), rnd(Mp, K), rnd(K)
    pos = torch.randperm(M * topk, device="cuda", generator=g).to(torch.int32)
    sc, ss = (torch.rand(M, n, device="cuda", generator=g).to(torch.bfloat16) for n in (topk - 1, 1))
    out = [(torch.empty_like(res), torch.empty(Mp, K, dtype=torch.int8, device="cuda"), torch.empty(Mp, device="cuda")) for _ in range(2)]
    for name, (h, xq, xs) in zip(("scmx_moe_combine", "scmx_moe_combine_blocked"), out):
        getattr(_lib.native(), name)(y, pos, sc, ss, res, w, 1e-6, h, xq, xs, M, Mp, K, topk)
    (h, xq, xs), (hb, xb, xsb) = out
    assert torch.equal(h, hb) and torch.equal(xs, xsb) and torch.equal(S.BlockedXq(xb.reshape(-1), Mp, K).rows(), xq)
