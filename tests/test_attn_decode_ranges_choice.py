"""Into how many ranges the decode attention cuts a cache, by its rows, heads and head dim: both sides of the measured lines."""
import pytest


@pytest.mark.parametrize("hq,hk,d,few,many", [(16, 8, 128, 3200, 4096), (16, 2, 128, 3200, 4096), (8, 4, 128, 6000, 12000),
                                              (4, 2, 128, 6000, 12000), (32, 8, 128, 3072, 3200), (16, 8, 64, 6000, 12000),
                                              (32, 8, 64, 3200, 6000), (8, 2, 64, 12000, 16000), (16, 8, 256, 3072, 3200),
                                              (8, 4, 256, 3200, 4096)])
def test_two_heads_a_reading_where_it_pays(hq, hk, d, few, many):
    from mxfp4_int8_m5_amd.sc_kernels import _decode_ranges
    assert [_decode_ranges(n, hq, hk, d) for n in (few, many)] == [16, 32]


@pytest.mark.parametrize("hq,hk,rows,ranges", [(16, 8, 512, 1), (16, 8, 513, 16), (24, 8, 12000, 16), (16, 16, 12000, 16), (40, 8, 12000, 16),
                                               (40, 8, 4000, 8), (64, 8, 1024, 1)])
def test_other_counts(hq, hk, rows, ranges):
    from mxfp4_int8_m5_amd.sc_kernels import _decode_ranges
    assert _decode_ranges(rows, hq, hk, 128) == ranges
