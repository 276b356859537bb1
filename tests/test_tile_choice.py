"""Which product kernel the size rules pick, without a GPU: the shapes that
tests/test_gpu_tile_choice.py runs each kernel at, so that a retuned rule cannot
take a kernel out of their reach unseen."""
import pytest

# nb, nv, ncouls, ngpown.  16 x 16 tiles: stages of 24 bands in a ring of six
# (23 to 25: one stage; 120, 121, 144, 145, 168, 169: five, six and seven
# stages), columns and G-vectors around 16
GRAM_16 = [
    (25, 2, 65, 33), (26, 2, 100, 64), (26, 2, 16, 33), (27, 2, 17, 1), (27, 2, 15, 17), (33, 2, 33, 15),
    (50, 2, 16, 16), (51, 2, 100, 31), (122, 2, 129, 16), (123, 2, 64, 47), (146, 2, 200, 15), (147, 2, 90, 48),
    (170, 2, 64, 49), (171, 2, 17, 1),
]
# 32 x 64 tiles: stages of 16 bands in a ring of three, columns around 32,
# G-vectors around 64
GRAM_32 = [
    (3, 2, 129, 33), (9, 2, 63, 64), (17, 2, 64, 63), (18, 2, 65, 65), (19, 2, 127, 96), (19, 2, 64, 97),
    (35, 2, 1000, 400), (50, 2, 1000, 700), (51, 2, 900, 321), (49, 2, 1500, 353), (102, 2, 700, 300),
]
# acht_n1_loc products of 64 x 128 tiles, the last tile short (at most 32
# columns) and whole: columns around 64, unoccupied bands around 128, G-vectors
# not in eights
ACHT_128_CUT = [
    (386, 2, 1001, 129), (387, 2, 1001, 193), (386, 3, 1001, 129), (386, 2, 1001, 160), (200, 3, 2003, 160),
    (131, 2, 2999, 32), (131, 2, 3000, 1),
]
ACHT_128 = [
    (514, 2, 1001, 128), (387, 2, 4093, 64), (257, 2, 2003, 128), (514, 2, 2003, 33), (387, 2, 4093, 33),
    (257, 2, 4093, 33), (200, 2, 2003, 127),
]
# Groups of bands in one launch, by their unoccupied bands: none, one, and
# around one stage of the 16 x 16 tile
GROUPS_16 = {"nv": 5, "unoccupied": [0, 1, 23, 24, 25, 60], "ncouls": 100, "ngpown": 33}


def gram(lib, nb, nv, nc, ng, groups=0, bands=0):
    return lib.gpp_test_gram_tile(nb, nv, nc, ng, groups, bands)


@pytest.mark.parametrize("tile,shapes", [(16016, GRAM_16), (32064, GRAM_32)])
def test_gram_tiles(gpplib, tile, shapes):
    assert [gram(gpplib, *s) for s in shapes] == [tile] * len(shapes)


def test_gram_tile_of_groups(gpplib):
    g = GROUPS_16
    nb = g["nv"] + sum(g["unoccupied"])
    assert gram(gpplib, nb, g["nv"], g["ncouls"], g["ngpown"], len(g["unoccupied"]), sum(g["unoccupied"])) == 16016


@pytest.mark.parametrize("tile,shapes", [(1064128, ACHT_128_CUT), (64128, ACHT_128)])
def test_acht_tiles(gpplib, tile, shapes):
    assert [gpplib.gpp_test_acht_tile(*s) for s in shapes] == [tile] * len(shapes)


def test_the_benchmark_shapes(gpplib):
    assert gram(gpplib, 512, 2, 800, 40) == 16016
    assert gram(gpplib, 512, 2, 4096, 409) == 64064
    assert gram(gpplib, 512, 2, 32768, 1638) in (64128, 128064)
    assert gpplib.gpp_test_acht_tile(512, 2, 4096, 409) == 1064128
