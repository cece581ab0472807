"""With weights unpacked to INT8 on every call (FUSE_UNPACK off), a prompt unpacks each matrix once: none is unpacked only to see which
layout its GEMM wants."""
import pytest
import torch

from tests.test_gpu_model import default_format_afterwards, make_tiny, make_tiny_moe   # noqa: F401 (a fixture for every test)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sparse,matrices", [(False, 4), (True, 2)])   # of a block, the experts apart
def test_one_unpack_a_matrix(sparse, matrices, monkeypatch):
    from mxfp4_int8_m5_amd import sc_kernels as S
    mod, args, state, packed = make_tiny_moe(4) if sparse else make_tiny(4, 2, 64)
    model = mod.FusedOlmoe(args, state, packed, tile=64) if sparse else mod.FusedQwen3(args, state, packed)
    ids = torch.randint(0, args.vocab_size, (45,), generator=torch.Generator().manual_seed(3)).cuda()
    want, seen, real = model.hidden(ids), [], S.unpack_i8
    monkeypatch.setattr(S, "FUSE_UNPACK", False)
    monkeypatch.setattr(S, "unpack_i8", lambda *a, **k: (seen.append(a[2:4]), real(*a, **k))[1])
    assert torch.equal(model.hidden(ids), want)
    assert len(seen) == matrices * args.num_hidden_layers
