"""The embedding rows a prompt starts from: indexing's own rules for the ids, and zero rows up to whole tiles."""
import pytest
import torch

from mxfp4_int8_m5_amd.fused_qwen3 import embed_rows

EMBED = torch.randn(300, 8, generator=torch.Generator().manual_seed(0)).to(torch.bfloat16)
MASK = torch.arange(300) % 7 == 0


@pytest.mark.parametrize("ids", [torch.tensor([5]), torch.tensor([-1, 0, -300, 299]), torch.arange(-128, 0, dtype=torch.int32),
                                 torch.arange(260).reshape(2, 130), torch.arange(10)[:0], MASK, MASK.to(torch.uint8)])
@pytest.mark.filterwarnings("ignore:indexing with dtype torch.uint8")
def test_rows_are_those_of_indexing(ids):
    want = EMBED[ids.reshape(-1)]
    h, L, Mp = embed_rows(EMBED, ids)
    assert L == want.shape[0] and Mp % 128 == 0 and 0 <= Mp - L < 128 and h.shape == (Mp, 8)
    assert torch.equal(h[:L], want) and not h[L:].any()


@pytest.mark.parametrize("bad", [300, -301])
def test_ids_beyond_the_vocabulary_are_refused(bad):
    with pytest.raises(IndexError):
        embed_rows(EMBED, torch.tensor([0, bad]))


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["cuda", "cpu"])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_rows_on_the_gpu(dtype, where):
    ids = torch.arange(-150, 150, dtype=dtype)
    h, L, Mp = embed_rows(EMBED.cuda(), ids.to(where))
    assert (L, Mp) == (300, 384) and torch.equal(h[:L].cpu(), EMBED[ids.long()]) and not h[L:].any()


def test_embedding_that_requires_grad():
    """A model built from named_parameters(): the kernels behind the embedding cut the graph, so nothing is lost here."""
    h, L, _ = embed_rows(EMBED.clone().requires_grad_(), torch.tensor([1, 2]))
    assert torch.equal(h[:L], EMBED[1:3])
