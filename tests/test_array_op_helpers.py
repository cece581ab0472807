"""The helpers around the kernels that a program may call itself: the ctypes side of the binding, and the rotary embedding and
cache append as array ops, which the fused kernels must agree with."""
import types

import pytest
import torch

import mxfp4_int8_m5_amd as scmx
from mxfp4_int8_m5_amd import fused_olmoe, fused_qwen3


def test_ctypes_calls_check_the_status():
    lib = scmx._lib
    with pytest.raises(ValueError, match="scmx_act_quant failed"):
        lib.call("scmx_act_quant", None, None, None, 4, 4, 128, None)
    assert lib.ptr(None) is None
    with pytest.raises(ValueError):
        lib.ptr(torch.zeros(4))


def test_cache_append():
    args = fused_qwen3.Qwen3Args(num_key_value_heads=2, head_dim=4)
    c = fused_qwen3.KVCache(args, 5, "cpu")
    a, b = torch.ones(2, 3, 4).to(torch.bfloat16), 2 * torch.ones(2, 2, 4).to(torch.bfloat16)
    c.update_and_fetch(a, 3 * a)
    k, v = c.update_and_fetch(b, 3 * b)
    assert c.offset == 5 and torch.equal(k, torch.cat([a, b], 1)) and torch.equal(v, 3 * k)
    with pytest.raises(ValueError):
        c.update_and_fetch(b, b)


@pytest.mark.gpu
@pytest.mark.parametrize("h,d,L,off", [(4, 64, 7, 0), (2, 128, 3, 11)])
def test_fused_norm_rope_append_against_the_array_ops(h, d, L, off):
    S = scmx.sc_kernels
    g = torch.Generator(device="cuda").manual_seed(d)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(torch.bfloat16)   # noqa: E731
    y, qn, kn = rnd(L, 3 * h * d), rnd(h * d), rnd(h * d)
    model = types.SimpleNamespace(inv_freq=1.0 / (1e4 ** (torch.arange(d // 2, device="cuda", dtype=torch.float32) / (d // 2))))
    rope = lambda x: fused_olmoe.FusedOlmoe.rope(model, x, off)   # noqa: E731
    args = fused_qwen3.Qwen3Args(num_key_value_heads=h, head_dim=d)
    one, two = (fused_qwen3.KVCache(args, 32) for _ in range(2))
    one.offset = off
    q, k, v = S.qkv_fullnorm_y(y, qn, kn, 1e-5, L, h, d)
    one.update_and_fetch(rope(k), v)
    qf = S.qkv_fullnorm_rope(y, qn, kn, 1e-5, L, h, d, two.k, two.v, off, model.inv_freq)
    close = lambda a, b: torch.testing.assert_close(a.float(), b.float(), rtol=2 ** -7, atol=2e-6 * float(b.abs().max()))   # noqa: E731
    close(qf, rope(q))   # float32 rotations through different sine and cosine routines, one rounding to bf16
    close(two.k, one.k)
    assert torch.equal(two.v, one.v)
    out = torch.empty((L, h * d), dtype=torch.int8, device="cuda"), torch.empty(L, dtype=torch.float32, device="cuda")
    x = y[:, :h * d].contiguous()
    scmx._lib.call("scmx_act_quant", scmx._lib.ptr(x), *map(scmx._lib.ptr, out), L, L, h * d, scmx._lib.stream())
    assert all(torch.equal(a, b) for a, b in zip(out, S.act_quant(x, L)))
