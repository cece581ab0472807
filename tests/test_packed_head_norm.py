"""The packed output head takes the final norm into its prologue only where the prologue reads that norm: without a GPU."""
import types

import pytest
import torch

from mxfp4_int8_m5_amd import fused_qwen3, sc_decode

K, N = 256, 32


def logits(norm, monkeypatch):
    """The decode step's head on one row -> the arguments its GEMV got."""
    seen = {}

    def gemv(x, *_, **kw):
        seen.update(kw, x=x)
        return torch.zeros(N)

    monkeypatch.setattr(sc_decode, "gemv", gemv)
    model = types.SimpleNamespace(norm=norm, eps=1e-6, lm_head=None)
    step = types.SimpleNamespace(f=model, head=True, packed_head=(None, None, None, N), head_fmt=None)
    h = torch.randn(1, K, generator=torch.Generator().manual_seed(0)).to(torch.bfloat16)
    assert fused_qwen3.DecodeQwen3._logits(step, h).shape == (1, N)
    return h, seen


def test_a_bf16_norm_runs_in_the_prologue(monkeypatch):
    w = torch.rand(K).to(torch.bfloat16)
    h, seen = logits(w, monkeypatch)
    assert seen["pro"] == 2 and seen["nw"] is w and seen["x"] is h


@pytest.mark.parametrize("kind", ["float32", "strided", "unaligned"])
def test_other_norms_run_in_front(kind, monkeypatch):
    w = torch.rand(2 * K).to(torch.bfloat16)
    w = {"float32": w[:K].float(), "strided": w[::2], "unaligned": w[1:K + 1]}[kind]
    h, seen = logits(w, monkeypatch)
    want = fused_qwen3.rms_norm(h, w, 1e-6)   # float32 for a float32 norm, which the GEMV refuses
    assert seen["pro"] == 1 and seen["x"].dtype == want.dtype and torch.equal(seen["x"], want)
