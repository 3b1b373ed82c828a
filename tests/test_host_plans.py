"""Rules that choose between kernels by sizes, on both sides of their borders, and the sizes that other tests rely on."""
import pytest

import test_gpu_small
from plan_query import ask

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
