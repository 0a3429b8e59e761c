"""Rules that choose between two ways of computing the same, beside what was measured on MI355X."""

import pytest

from petals_amd.ops.fused_decode import norm_within

# k, n, whether sums of squares are given, and by rows: us with the norm ahead of the product and within
NORMS = [
    (512, 1024, False, {1: (5.4, 3.7), 4: (5.8, 5.1), 6: (5.9, 6.1)}),
    (2048, 2560, False, {1: (7.2, 5.4), 4: (7.5, 7.2), 5: (7.6, 7.8), 8: (8.1, 9.6)}),
    (2048, 6144, False, {1: (8.8, 7.1), 3: (9.1, 8.7), 5: (9.4, 10.1)}),
    (4096, 3072, False, {1: (9.0, 7.5), 3: (9.3, 9.2), 4: (9.4, 10.0)}),
    (4096, 6144, False, {1: (13.7, 11.5), 2: (13.8, 12.7), 4: (14.1, 14.3), 8: (15.3, 17.7)}),
    (4096, 12288, False, {1: (21.2, 19.6), 2: (21.4, 22.4), 4: (21.6, 25.2)}),
    (5120, 7680, False, {1: (19.5, 19.1), 2: (19.7, 21.1)}),
    (5120, 15360, False, {2: (30.3, 33.8)}),
    (8192, 2560, False, {1: (13.2, 11.4), 3: (13.6, 13.7), 4: (13.6, 14.8)}),
    (8192, 5120, False, {1: (19.9, 20.4), 4: (20.3, 26.0)}),
    (8192, 10240, False, {1: (31.5, 33.8), 4: (32.4, 43.0)}),
    (16384, 18432, False, {1: (101.4, 113.2), 4: (107.6, 153.3)}),
    (1024, 8192, True, {1: (10.0, 8.2), 5: (10.8, 10.4), 8: (11.5, 12.2)}),
    (2048, 11264, True, {1: (15.6, 13.0), 5: (16.4, 15.4), 8: (17.2, 17.6)}),
    (4096, 5504, True, {1: (15.9, 13.3), 5: (17.0, 15.4)}),
    (4096, 28672, True, {1: (44.1, 41.5), 2: (44.7, 43.3), 3: (45.2, 47.7), 8: (49.9, 61.3)}),
    (5120, 27648, True, {2: (52.9, 51.4), 3: (54.4, 58.1)}),
    (8192, 57344, True, {1: (153.7, 151.2), 3: (166.6, 174.0), 8: (190.3, 224.0)}),
    (16384, 106496, True, {1: (549.7, 545.9), 4: (629.1, 708.8)}),
]


@pytest.mark.parametrize("k,n,summed,times", NORMS)
def test_norms_within_products(k, n, summed, times):
    """Within where it is faster, ahead where it is not, but for differences of 3%."""
    for rows, (ahead, within) in times.items():
        if abs(within - ahead) > 0.03 * ahead:
            assert norm_within(rows, k, n, summed) == (within < ahead), rows
