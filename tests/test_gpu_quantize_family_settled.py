"""The family quantizer settles most trials on a bounded error first: weights on which it cannot (equal errors of several multipliers or
bases, blocks and rows near the ends of the float32 range, zeros, infinities) next to ordinary ones, bit for bit against the oracle."""
import numpy as np
import pytest
import torch

from oracle import family
from tests.util import dev, host

pytestmark = pytest.mark.gpu


def rows(rng, k, block, mults):
    """[19, k] float32: ordinary rows and rows that hold the cases above."""
    w = (rng.standard_normal((19, k)) * 0.02 * np.exp(0.4 * rng.standard_normal(k))).astype(np.float32)
    levels = np.array([0, 1, 2, 3, 4, 6, 8, 12], np.float32)
    m = np.repeat(rng.choice(mults, (4, k // block)), block, 1)
    w[0:4] = rng.choice(levels, (4, k)) * rng.choice([-1, 1], (4, k)) * m * 2.0 ** -7      # exact at one base, often at several scales
    w[1] = np.where(rng.random(k) < 0.5, 0, w[1])
    w[2, :] = 0.125                                                                        # equal weights: equal errors
    w[3] = np.rint(w[3] * 64) / 64
    w[4, :5 * block] = 0                                                                   # zero blocks
    w[5] *= 1e-30
    w[6] *= 1e30
    w[7, block:2 * block] *= 1e-12                                                         # one tiny block: the row is summed as before
    w[8] = 0
    w[9, 3] = 40.0                                                                         # an outlier: the other blocks clip nowhere
    w[10] = np.float32(1e-42)
    w[11, ::block] = -0.0
    w[12] = rng.integers(-12, 13, k) * 0.5
    w[13] = np.abs(w[13])
    return w


@pytest.mark.parametrize("name", ["e2m1/B16/M1..10", "e2m1/B32/pow2", "e2m1/B16/M3..10"])
@pytest.mark.parametrize("k,copies", [(128, 1), (1024, 1), (896, 12), (2048, 40)])   # side by side, and a thread per block
@pytest.mark.parametrize("bf", [False, True])
def test_equals_the_oracle(name, k, copies, bf):
    from mxfp4_int8_m5_amd import pack_format
    fam = family.member(name)
    rng = np.random.default_rng(k + copies)
    w = rows(rng, k, fam.block, fam.mults)
    t = torch.from_numpy(w)
    if bf:
        t = t.to(torch.bfloat16)
        w = t.float().numpy()
    codes, bc, ws = pack_format.pack_matrix(t.cuda().repeat(copies, 1), name)[:3]
    _, q, base, bscale = family.quantize(w, fam)
    fmt = fam.storage()
    want = family.pack_parts(q, base, bscale, fmt)
    n = len(w)
    for got, ref in zip((codes, bc, ws), want):
        got = host(got).reshape(copies, n, -1)
        ref = np.ascontiguousarray(ref).view(got.dtype).reshape(n, -1)
        for c in range(copies):
            assert np.array_equal(got[c], ref), [i for i in range(n) if not np.array_equal(got[c][i], ref[i])]


def test_infinities_and_nan_take_the_evaluation_of_every_trial():
    """No value of theirs is defined: the call returns, and rows beside them are what they are alone."""
    from mxfp4_int8_m5_amd import pack_format
    rng = np.random.default_rng(5)
    w = rows(rng, 256, 16, np.arange(1, 11))
    alone = pack_format.pack_matrix(torch.from_numpy(w).cuda(), "e2m1/B16/M1..10")[:3]
    w2 = np.repeat(w, 2, 0)
    w2[1::2, 7] = np.tile([np.inf, np.nan, -np.inf], 7)[:19]
    both = pack_format.pack_matrix(torch.from_numpy(w2).cuda(), "e2m1/B16/M1..10")[:3]
    for a, b in zip(alone, both):
        assert torch.equal(a.reshape(19, -1), b.reshape(38, -1)[::2])
