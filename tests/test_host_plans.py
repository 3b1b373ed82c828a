"""Rules that choose between kernels by sizes, on both sides of their borders, and the sizes that other tests rely on."""
import pytest

import test_gpu_block_tiles
import test_gpu_small
from plan_query import TILES, ask

Q4, Q8 = 18, 34


def small(dim, ff, heads, layers, vocab, block=Q4):
    return ask([("small", dim, ff, heads, dim // heads, layers, vocab, block)])[0]


@pytest.mark.parametrize("block", [Q4, Q8])
@pytest.mark.parametrize("shape,own", [
    # partial sums are faster up to 288 columns ...
    ((64, 160, 1, 4, 512), 1), ((256, 704, 4, 8, 32000), 1), ((256, 704, 4, 2, 64000), 1), ((256, 4096, 4, 4, 512), 2), ((288, 768, 9, 6, 32000), 1),
    # ... and were 1 to 6 % slower in some of these
    ((320, 4000, 5, 4, 512), 0), ((384, 2048, 12, 4, 512), 0), ((384, 1024, 6, 6, 32000), 0), ((448, 1216, 7, 4, 32000), 0),
    ((512, 1376, 4, 6, 4096), 0), ((512, 704, 4, 4, 512), 0), ((768, 2048, 12, 12, 512), 0),
    # more feed-forward blocks than two for each workgroup
    ((256, 4128, 4, 2, 512), 0),
])
def test_partial_sums_of_small_models(shape, own, block):
    wgs, got, _ = small(*shape, block)
    assert wgs and got == own


def test_workgroups_of_a_small_models_launch():
    """every head and, with partial sums, every workgroup's feed-forward blocks have a workgroup; a launch takes a quarter of 256 CUs at most"""
    for dim in range(32, 1025, 32):
        for heads in {dim // r for r in (32, 64, 128) if dim % r == 0}:
            for ff in (32, 96, 704, 2016, 2048, 2080, 4064, 4096, 4128, 8192):
                for vocab in (300, 32000, 128256):
                    wgs, own, _ = small(dim, ff, heads, 2, vocab)
                    if wgs:
                        assert heads <= wgs <= 64
                        assert not own or (-(-ff // 32 // own) <= wgs and own & (own - 1) == 0 and dim * max(own, dim // heads // 32) <= 4 * 512)


@pytest.mark.parametrize("shape,launch", [
    # a narrow model's large vocabulary: the chain copies its logits (one layer 106 us, the launch 87)
    ((256, 704, 4, 1, 128256), True), ((128, 352, 2, 1, 128256), True), ((192, 512, 3, 2, 100000), True), ((256, 704, 4, 2, 128256), True),
    # a wider one's products are too much for a quarter of the CUs
    ((640, 1728, 10, 4, 128256), False), ((1024, 64, 16, 1, 32000), False), ((1024, 2816, 16, 1, 128256), False), ((1024, 8160, 8, 2, 1000), False),
])
@pytest.mark.parametrize("block", [Q4, Q8])
def test_small_models_beside_the_operator_chain(shape, launch, block):
    assert (small(*shape, block)[0] > 0) == launch


def test_small_shapes_of_the_gpu_tests_take_the_ways_they_are_there_for():
    for name, c in test_gpu_small.SHAPES.items():
        for block in (Q4, Q8):
            wgs, own, _ = small(c["dim"], c["ff"], c["heads"], c["layers"], c["vocab"], block)
            assert (wgs == 0) == (name in test_gpu_small.CHAIN), name
            if wgs:
                assert own == {"three blocks a row": 1, "one head, one block": 1, "head of 128": 1, "a block a workgroup": 1, "workgroups without blocks": 1,
                               "widest with partial sums": 1, "two columns a lane": 2, "two blocks a workgroup": 2}.get(name, 0), name


def up(v, a):
    return (v + a - 1) // a * a


def dense_plans(shapes):
    """of gate and up, and of down, in a feed-forward of (width, ff) and n tokens: tile, slices, K steps of a slice, units of 32 tokens in the rest"""
    asked = []
    for width, ff, n in shapes:
        rows = up(2 * up(ff, 16), 128)
        asked += [("product", rows, n, up(width, 64), 1), ("product", width, n, rows // 2, 4 if n <= 1024 else 1)]
    for (_, rows, n, columns, _), (tile, slices) in zip(asked, ask(asked)):
        yield TILES[tile], slices, columns // 64, -(-(n % int(TILES[tile][4:])) // 32)


def test_dense_shapes_of_the_gpu_tests_reach_every_tile():
    """with every rest of whole units: each is a loop of its own.  A plan that moves has to move the shapes too"""
    plans = list(dense_plans(test_gpu_block_tiles.DENSE))
    dense, store = plans[::2], plans[1::2]
    for tile, units in ("256x128", 4), ("256x160", 5), ("256x192", 6):
        assert {p[3] for p in dense if p[0] == tile} >= set(range(units)), tile
    assert {p[3] for p in dense if p[0] == "256x256"} >= {0, 1, 2, 5, 8}      # its rests share one loop; a whole 128 tokens missing, and less
    for tile, steps in ("128x128", 1), ("256x128", 3), ("256x160", 3), ("256x192", 2), ("256x256", 2):
        assert min(p[2] for p in dense if p[0] == tile) <= steps, tile
    for tile, slices in ("128x128", {1, 2, 3, 4}), ("256x128", {1, 2, 3, 4}), ("256x160", {1, 2, 4}), ("256x192", {1, 2}), ("256x256", {1}):
        assert {p[1] for p in store if p[0] == tile} >= slices, tile
    for tile in "128x128", "256x128", "256x160", "256x192":
        assert any(p[0] == tile and p[1] > 1 and p[2] % p[1] for p in store), tile      # a last slice that is shorter


def experts(width, ff, n, count, top):
    rows = up(2 * up(ff, 16), 128)
    gate_up, down, by_expert = ask([("experts", n, count, top, rows, up(width, 64), up(width, 128), rows // 2)])[0]
    return TILES[gate_up], TILES[down], bool(by_expert)


def test_expert_shapes_of_the_gpu_tests_reach_every_tile_and_order():
    seen = set()
    for width, ff, n, count, top in test_gpu_block_tiles.EXPERTS:
        gate_up, down, by_expert = experts(width, ff, n, count, top)
        several = n * top > 128 * count
        seen |= {("gate_up", gate_up, by_expert, several), ("down", down, several)}
    assert seen == {("gate_up", t, o, s) for t in ("128x128", "256x128") for o in (False, True) for s in (False, True)} | {
        ("down", t, s) for t in ("128x128", "256x128") for s in (False, True)}


@pytest.mark.parametrize("width,ff,count,top,n,want", [
    # small experts: 128 x 128 (256 rows x 128 or 160 tokens were 3 to 8 % of a prompt slower)
    (1024, 512, 8, 2, 100, ("128x128", "128x128", False)), (1024, 512, 8, 2, 777, ("128x128", "128x128", False)), (512, 512, 16, 4, 512, ("128x128", "128x128", False)),
    (1024, 512, 32, 4, 512, ("128x128", "128x128", False)),
    # large ones: 256 x 128, a row tile after the other (an expert after the other up to 10 % slower)
    (4096, 7168, 8, 2, 512, ("256x128", "256x128", False)), (4096, 7168, 8, 2, 1300, ("256x128", "256x128", False)), (8192, 2048, 16, 2, 640, ("256x128", "256x128", False)),
    (2048, 1024, 32, 4, 900, ("256x128", "128x128", False)), (4096, 1024, 64, 8, 512, ("256x128", "256x128", False)), (4096, 1024, 64, 8, 2048, ("256x128", "256x128", False)),
    # few tokens of many experts: an expert after the other
    (4096, 1024, 64, 8, 100, ("256x128", "256x128", True)), (4096, 768, 128, 8, 640, ("256x128", "256x128", True)),
])
def test_tiles_of_chosen_experts(width, ff, count, top, n, want):
    assert experts(width, ff, n, count, top) == want


@pytest.mark.parametrize("rows,n,columns,slices,want", [
    # few workgroups take as long a step as they load: 128 x 128 (256 x 128 1.2 times as long)
    (5248, 100, 5120, 1, ("128x128", 1)), (5248, 256, 5120, 1, ("128x128", 1)), (3200, 128, 3072, 1, ("128x128", 1)), (7296, 512, 7168, 1, ("128x128", 1)),
    # but with a rest that runs ahead of the other tiles of its rows
    (2112, 777, 4096, 1, ("256x128", 1)), (5248, 900, 5120, 1, ("256x128", 1)),
    # slices of long rows in tiles of 160 tokens took 1.6 times what they were thought to
    (7168, 460, 19392, 4, ("256x128", 2)), (7168, 512, 18432, 4, ("256x128", 2)),
    # large products
    (18560, 500, 4096, 1, ("256x192", 1)), (13600, 2048, 4096, 1, ("256x256", 1)), (8848, 1000, 2048, 1, ("256x160", 1)),
])
def test_tiles_of_products(rows, n, columns, slices, want):
    tile, got = ask([("product", rows, n, columns, slices)])[0]
    assert (TILES[tile], got) == want
