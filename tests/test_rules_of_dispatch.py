"""Rules that choose between two ways of computing the same, beside what was measured on MI355X."""

import csv
import os

import pytest

from petals_amd.ops.fused_decode import norm_within
from petals_amd.ops.prompt_grad import takes_gemm, takes_wide_gemm

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


# k, n, what follows or from which side, and by rows: us by the library (with what follows) and by gemm.hip
PRODUCTS = [
    (2048, 2560, "",
     {16: (10.9, 11.1), 64: (13.7, 11.5), 128: (18.0, 12.5), 256: (13.8, 16.3), 384: (13.9, 19.9), 758: (18.9, 18.8)}),
    (2048, 2048, "",
     {16: (8.4, 10.4), 64: (12.8, 10.9), 128: (10.5, 11.7), 256: (12.1, 14.9), 384: (13.1, 17.5), 758: (16.7, 17.7)}),
    (2048, 11264, "fused",
     {16: (17.6, 16.7), 64: (19.9, 19.2), 128: (25.2, 29.3), 256: (34.4, 27.3), 384: (37.9, 33.6), 758: (45.5, 46.2)}),
    (5632, 2048, "added",
     {16: (25.5, 15.5), 64: (43.5, 17.0), 128: (28.1, 19.3), 256: (32.4, 20.2), 384: (41.6, 22.4), 758: (46.5, 31.7)}),
    (4096, 12288, "",
     {16: (25.8, 24.3), 64: (33.8, 27.6), 128: (39.9, 32.7), 256: (55.0, 43.0), 384: (58.7, 57.2), 758: (72.5, 84.6)}),
    (4096, 6144, "",
     {16: (22.6, 17.0), 64: (28.2, 19.8), 128: (38.3, 21.4), 256: (47.6, 28.9), 384: (40.5, 36.0), 758: (53.3, 54.6)}),
    (4096, 28672, "fused",
     {16: (56.2, 48.9), 64: (48.8, 51.8), 128: (56.5, 58.3), 256: (78.0, 73.2), 384: (90.2, 108), 758: (167, 172)}),
    (5120, 27648, "fused",
     {16: (70.9, 57.3), 64: (59.4, 59.7), 128: (70.4, 76.0), 256: (92.4, 91.1), 384: (108, 131), 758: (200, 211)}),
    (8192, 10240, "",
     {16: (48.0, 36.8), 64: (63.5, 39.7), 128: (75.6, 44.2), 256: (111, 62.4), 384: (94.1, 83.4), 758: (133, 119)}),
    (8192, 57344, "fused",
     {16: (162, 168), 64: (166, 170), 128: (178, 177), 256: (224, 281), 384: (349, 375), 758: (616, 652)}),
    (16384, 106496, "fused", {16: (597, 635), 64: (766, 644), 128: (861, 770)}),
    (8192, 14336, "fused", {64: (66.6, 51.9), 128: (78.6, 59.5), 256: (97.6, 98.8), 384: (109, 135), 512: (135, 124)}),
    (28672, 8192, "added",
     {16: (134, 85.6), 64: (199, 88.9), 128: (203, 97.0), 256: (287, 134), 384: (197, 209), 758: (321, 398)}),
    (1024, 3072, "",
     {16: (7.5, 9.8), 64: (10.9, 10.2), 128: (10.9, 10.9), 256: (9.5, 12.5), 384: (12.4, 10.6), 758: (17.1, 11.9)}),
    (4096, 16384, "fused",
     {16: (29.1, 29.8), 64: (34.3, 32.6), 128: (46.6, 37.5), 256: (59.0, 47.4), 384: (60.9, 65.7), 758: (98.3, 112)}),
    (4544, 18176, "fused",
     {16: (46.0, 33.0), 64: (53.2, 36.2), 128: (56.3, 43.6), 256: (78.4, 65.6), 384: (78.0, 73.0), 758: (118, 138)}),
    (2560, 2048, "transposed",
     {16: (8.1, 11.1), 64: (9.9, 11.8), 128: (9.4, 12.7), 256: (10.6, 16.2), 384: (11.9, 19.6), 758: (15.1, 19.8)}),
    (11264, 2048, "transposed",
     {16: (16.7, 20.3), 64: (30.0, 20.5), 128: (26.6, 22.3), 256: (35.9, 25.5), 384: (44.3, 31.9), 758: (57.5, 46.0)}),
    (12288, 4096, "transposed",
     {16: (20.8, 28.2), 64: (35.3, 30.9), 128: (63.8, 31.3), 256: (51.4, 40.9), 384: (65.2, 51.4), 758: (88.5, 92.9)}),
    (4096, 4096, "transposed",
     {16: (14.9, 15.7), 64: (14.6, 16.4), 128: (23.8, 18.5), 256: (22.0, 21.2), 384: (24.5, 27.5), 758: (32.4, 36.5)}),
    (16384, 16384, "transposed", {16: (97, 140), 64: (105, 147), 128: (137, 153)}),
    (32768, 8192, "transposed", {16: (100, 132), 64: (152, 136), 283: (333, 213), 384: (218, 238)}),
    (106496, 16384, "transposed", {128: (632, 601), 129: (666, 1079), 192: (775, 838)}),
    (22016, 4096, "transposed",
     {16: (56.4, 44.8), 64: (134, 48.0), 128: (114, 50.8), 256: (153, 66.0), 384: (230, 82.6), 758: (230, 160)}),
    (4096, 11008, "transposed",
     {16: (25.2, 24.2), 64: (26.6, 26.7), 128: (30.7, 31.1), 256: (47.2, 41.4), 384: (48.1, 51.4), 758: (62.8, 74.6)}),
    (8192, 8192, "transposed",
     {16: (28.0, 33.1), 64: (31.4, 35.3), 128: (46.0, 41.8), 256: (74.4, 52.3), 384: (60.9, 71.7), 758: (93.1, 113)}),
    (57344, 8192, "transposed",
     {16: (157, 164), 64: (267, 170), 128: (298, 184), 256: (455, 267), 384: (370, 417), 758: (557, 755)}),
    (15360, 5120, "transposed",
     {16: (35.4, 35.9), 64: (51.9, 38.7), 128: (80.9, 43.2), 256: (131, 58.9), 384: (97.8, 73.9), 758: (134, 121)}),
]


@pytest.mark.parametrize("k,n,kind,times", PRODUCTS)
def test_products_of_prompts(k, n, kind, times):
    """What is taken is slower by less than the 10 us that the library's call takes longer on the host;
    few rows and long sums, which the kernel is for, are taken."""
    for rows, (library, kernel) in times.items():
        taken = takes_gemm(rows, k, n, **({kind: True} if kind else {}))
        assert kernel <= library + 10 or not taken, rows
        if k >= 5 * n and kernel < 0.8 * library:
            assert taken, rows
    if k < 3000 and n < 3000 and not kind:  # prompts of 300 rows and more are bound by the kernels
        assert all(kernel <= library + 1.5 for rows, (library, kernel) in times.items() if rows > 300 and takes_gemm(rows, k, n))


# the same for the tiles of 256 columns that four waves have, where the library had the product
WIDE = [
    (4096, 12288, "", {192: (59.2, 46.1), 512: (59.0, 62.1), 758: (72.7, 66.3), 1024: (88.3, 91.5), 4096: (317, 329)}),
    (4096, 22016, "followed", {512: (104, 98), 1024: (187, 169), 2048: (385, 311), 4096: (740, 604)}),
    (4096, 28672, "followed", {512: (116, 109), 1024: (223, 205), 2048: (454, 394), 4096: (842, 757)}),
    (8192, 57344, "followed", {512: (441, 412), 1024: (846, 767), 2048: (1573, 1463), 4096: (3084, 2858)}),
    (8192, 10240, "", {283: (82.2, 68.1), 512: (110, 82.6), 758: (135, 114), 1200: (194, 188)}),
    (16384, 4096, "followed", {512: (145, 73), 1024: (177, 126), 2048: (261, 231), 4096: (426, 425)}),
    (18176, 4544, "", {512: (221, 87), 1024: (257, 147), 2048: (373, 296), 4096: (978, 540)}),
    (22016, 4096, "transposed", {512: (229, 88.5), 758: (230, 119), 1500: (387, 216), 4096: (540, 620)}),
    (12288, 4096, "transposed", {758: (91.3, 73.1), 1024: (112, 89.9), 4096: (271, 296)}),
    (8192, 8192, "transposed", {512: (76.7, 70.6), 1024: (113, 114), 2048: (174, 195), 4096: (357, 397)}),
    (4096, 11008, "transposed", {283: (48.4, 43.5), 512: (53.3, 58.4), 1024: (76.0, 92.4)}),
    (8192, 28672, "transposed", {448: (165, 187)}),
    (4544, 18176, "transposed", {192: (59, 53), 512: (81, 96), 758: (98, 112), 1200: (256, 185), 1500: (188, 224), 2048: (313, 286)}),
]


@pytest.mark.parametrize("k,n,kind,times", WIDE)
def test_wide_products(k, n, kind, times):
    """Taken where it is faster, and nowhere where it is slower by more than 6%, which is what noise and the host make up."""
    for rows, (library, kernel) in times.items():
        taken = takes_wide_gemm(rows, k, n, **({kind: True} if kind else {}))
        assert taken or kernel > 0.94 * library, rows
        assert not taken or kernel < 1.06 * library, rows


MEASURED = os.path.join(os.path.dirname(__file__), os.pardir, "profiles", "prompt_products_wide.csv")


@pytest.mark.skipif(not os.path.exists(MEASURED), reason="what was measured is not here")
def test_rules_beside_all_that_was_measured():
    """What large products take is no more than 7% slower anywhere, and 10% faster in the mean; what they leave is no
    faster in the mean. What the others take is slower by less than the 10 us that the library's call takes longer on the
    host, but for 3%, and the tile that is chosen is 2% slower than the best one in the mean."""
    with open(MEASURED) as f:
        products = [(r["follows"], *(int(r[c]) for c in ("rows", "k", "n", "transposed")), r) for r in csv.DictReader(f)]
    assert len(products) > 1500
    taken, left, chosen = [], [], {True: [], False: []}
    for follows, m, k, n, transposed, r in products:
        library, kernel, tiles = float(r["library"]), float(r["kernel"]), [float(r[f"tile{i}"]) for i in range(9)]
        chosen[k * n <= 25 << 20].append(kernel / min(t for t in tiles if t))
        if takes_gemm(m, k, n, bool(transposed), fused=follows in ("gelu", "swiglu"), added=follows == "residual"):
            assert kernel <= 1.03 * library + 10, r
        elif takes_wide_gemm(m, k, n, bool(transposed), followed=follows in ("residual", "swiglu"), gelu=follows == "gelu"):
            assert kernel <= 1.07 * library, r
            taken.append(kernel / library)
        elif m > 128 and k * n > 25 << 20:
            left.append(kernel / library)
    assert sum(taken) < 0.9 * len(taken) and sum(left) > len(left)
    for which in chosen.values():
        assert sum(which) < 1.02 * len(which)


@pytest.mark.parametrize("m,k,n", [(128, 8192, 8192), (700, 2048, 11264), (758, 2048, 2560), (512, 16384, 53248), (1 << 19, 4096, 4096)])
def test_what_wide_products_leave(m, k, n):
    """Few rows, small matrices, what offsets of 32 bits don't reach."""
    assert not takes_wide_gemm(m, k, n, followed=True)


@pytest.mark.parametrize(
    "m,k,n,taken",
    [
        (758, 4096, 22016, True), (768, 4096, 22016, True), (512, 4096, 22016, False), (769, 4096, 22016, False),  # 258, 172 and 344 tiles
        (4097, 4096, 4096, True), (4096, 4096, 4096, False), (4353, 4096, 4096, False),  # 272, 256, 288
        (1700, 3584, 18944, True), (1536, 3584, 18944, False),  # 518, 444
        (1537, 4096, 28160, False),  # 770
        (6600, 2048, 2560, False), (33000, 512, 512, False),  # 260, 258 of small matrices, which nothing is known of
    ],
)
@pytest.mark.parametrize("transposed", [False, True])
def test_few_tiles_of_the_library_left_over(m, k, n, taken, transposed):
    """After one or two turns of all compute units they cost it another one, whatever the matrix."""
    assert takes_wide_gemm(m, k, n, transposed) == taken


@pytest.mark.parametrize("k,n", [(4544, 18176), (4160, 13120), (7232, 28864)])
def test_turns_of_the_library_with_little_work(k, n):
    """Sizes that it has no good kernel for and many columns: the rows at which its tiles leave a fifth of the turns idle."""
    columns = -(-n // 256)
    for rows in range(513, 8192, 101):
        tiles = -(-rows // 256) * columns
        turns = -(-tiles // 256)
        taken = turns > 3 or turns > 1 and (tiles < 0.8 * turns * 256 or 0 < tiles % 256 <= 20)
        for transposed in (False, True):
            assert takes_wide_gemm(rows, k, n, transposed) == taken, rows
