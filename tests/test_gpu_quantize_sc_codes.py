"""The published format's codes leave through the FP4 conversion: weights on every midpoint and one unit in the last place either side
of it, both signs, zeros of both signs, exponents near the ends of the range, against the host's rounding."""
import numpy as np
import pytest
import torch

from oracle import layout
from tests.util import dev, host, product_format

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bf", [False, True])
@pytest.mark.parametrize("block", [16, 32])
@pytest.mark.parametrize("n,k", [(3, 128), (40, 1024), (700, 896)])
def test_midpoints(n, k, block, bf):
    from mxfp4_int8_m5_amd import sc_format as F
    rng = np.random.default_rng(n + k + block)
    mids = np.array([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0, 6.0, 0.5, 0.0], np.float32)
    w = rng.standard_normal((n, k)).astype(np.float32)
    pick = rng.random((n, k)) < 0.6
    w = np.where(pick, rng.choice(mids, (n, k)) * rng.choice(np.float32([-1, 1]), (n, k)), w).astype(np.float32)
    step = rng.integers(-1, 2, (n, k)) * (w != 0)
    w = (w.view(np.int32) + np.where(pick, step, 0).astype(np.int32)).view(np.float32)
    w[:, ::block] = 6.0                                            # the block's exponent is that of the midpoints' scale
    w[0, 5] = -0.0
    w *= np.exp2(rng.choice([-110, -90, -20, 0, 30, 110] if not bf else [-90, -20, 0, 30], (n, 1))).astype(np.float32)
    t = torch.from_numpy(w)
    if bf:
        t = t.to(torch.bfloat16)
        w = t.float().numpy()
    codes, bc, ws, q = F.quantize(t.cuda(), product_format(layout.Format(block=block)))
    c0, b0, s0, q0 = layout.quantize(w.astype(np.float64), layout.Format(block=block))
    assert np.array_equal(host(ws), s0) and np.array_equal(host(bc), b0)
    assert np.array_equal(host(codes).view(np.uint32), c0) and np.array_equal(host(q), q0)


@pytest.mark.parametrize("block", [16, 32])
@pytest.mark.parametrize("n,k", [(3, 128), (40, 1024), (700, 896)])
def test_bf16_trials(n, k, block):
    """Exponents searched with half-precision differences: weights far below their block's largest (down to where half precision has
    no more bits, and below), on the levels of the three exponents tried, saturating, and blocks of equal magnitudes."""
    from mxfp4_int8_m5_amd import sc_format as F
    rng = np.random.default_rng(n * k + block)
    nb = k // block
    w = rng.standard_normal((n, nb, block)).astype(np.float32)
    w *= np.exp2(-rng.integers(0, 30, w.shape)).astype(np.float32)
    levels = np.array([0.125, 0.25, 0.375, 0.5, 0.75, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, 7.96875], np.float32)
    pick = rng.random(w.shape) < rng.choice([0.0, 0.3, 0.9], (n, nb, 1))
    w = np.where(pick, rng.choice(levels, w.shape) * rng.choice(np.float32([-1, 1]), w.shape), w).astype(np.float32)
    w[..., 0] = rng.choice(np.float32([4.0, 5.0, 6.0, 6.96875, 7.0, 7.96875]), (n, nb))
    same = rng.random((n, nb)) < 0.2
    w[same] = w[same][:, :1]
    w[rng.random((n, nb)) < 0.05] = 0.0
    w *= np.exp2(rng.integers(-3, 4, (n, nb, 1)) + rng.choice([-100, -20, 0, 30, 100], (n, 1, 1))).astype(np.float32)
    t = torch.from_numpy(w.reshape(n, k)).to(torch.bfloat16)
    codes, bc, ws, q = F.quantize(t.cuda(), product_format(layout.Format(block=block)))
    c0, b0, s0, q0 = layout.quantize(t.float().numpy().astype(np.float64), layout.Format(block=block))
    assert np.array_equal(host(ws), s0) and np.array_equal(host(bc), b0)
    assert np.array_equal(host(codes).view(np.uint32), c0) and np.array_equal(host(q), q0)
