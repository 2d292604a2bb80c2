"""The chunk length that the decoding drop-ins choose."""
import pytest

from tritonops_amd import _lib


@pytest.fixture(scope="module")
def choose():
    return _lib.load().mi_decode_choose_split


def test_bounds_of_the_choice(choose):
    for batch in (1, 3, 64, 4096):
        for units in (1, 8, 33, 512):
            for bound in (1, 64, 2048, 2049, 16384, 65537, 1 << 20, (1 << 31) - 1):
                t = choose(batch, units, bound, 256)
                assert t in (64, 128, 256, 512, 1024, 2048)
    assert choose(0, 8, 100, 256) == choose(1, 8, 0, 256) == 64
    assert choose(1, 8, 8192, 0) == choose(1, 8, 8192, 256)


@pytest.mark.parametrize("args,want", [((1, 8, 2048), 64), ((1, 8, 2049), 128), ((1, 1, 16385), 256), ((1, 1, 65537), 512),
                                       ((10, 8, 2048), 64), ((64, 8, 1024), 256), ((4, 8, 8192), 128), ((32, 2, 8192), 256),
                                       ((64, 8, 32768), 2048)])
def test_chunks_grow_with_the_work(choose, args, want):
    assert choose(*args, 256) == want
