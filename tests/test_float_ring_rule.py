"""Which float products go through the LDS ring, and with which tile: the sizes at which both sides were measured."""
import ctypes

import pytest


@pytest.fixture(scope="module")
def shape():
    from minivllm_amd.csrc import build
    return ctypes.CDLL(build.find_library("f32") or build.build("f32")).mv_gemm_ref_ring_shape


@pytest.mark.parametrize("size", [(224, 4096, 1024), (224, 1024, 3072), (16, 4096, 1024), (16, 151936, 1024), (500, 1024, 128), (200, 4096, 128),
                                  (64, 16384, 128), (1000, 1024, 256), (4096, 1024, 256), (4096, 1024, 512), (8192, 4096, 512),
                                  (200, 151936, 256)])
def test_through_the_ring(shape, size):
    assert shape(*size) in (22, 24, 44)


@pytest.mark.parametrize("size", [(1, 1024, 3072), (16, 1024, 3072), (224, 4096, 1000), (224, 4096, 64), (0, 4096, 1024),
                                  (2048, 1024, 128), (4096, 1024, 128), (200, 151936, 128)])
def test_straight_from_the_caches(shape, size):
    assert shape(*size) == 0


def test_tiles_whose_rounds_take_the_least(shape):
    assert [shape(*s) for s in [(224, 4096, 1024), (224, 6144, 1024), (224, 1024, 3072), (1024, 24576, 4096)]] == [44, 24, 22, 44]
