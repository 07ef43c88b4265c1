"""Which bfloat16 products the kernel takes whose waves split K: sizes at which both sides were measured."""
import ctypes

import pytest


@pytest.fixture(scope="module")
def shape():
    from minivllm_amd.csrc import build
    return ctypes.CDLL(build.find_library("bf16") or build.build("bf16")).mv_gemm_deep_shape


@pytest.mark.parametrize("rows, n, k, gated", [(9, 256, 4096, 0), (800, 512, 2048, 0), (500, 256, 4096, 0), (300, 576, 4096, 0), (200, 1024, 4096, 0),
                                               (64, 768, 8192, 0), (96, 768, 8192, 0), (500, 1024, 3072, 0), (128, 4096, 1024, 0),
                                               (32, 16384, 512, 0), (64, 4096, 512, 0), (32, 8192, 512, 1), (500, 1024, 8192, 1), (800, 512, 4096, 1)])
def test_served(shape, rows, n, k, gated):
    assert shape(rows, n, k, gated) != 0


@pytest.mark.parametrize("rows, n, k, gated", [(800, 256, 4096, 0), (500, 576, 4096, 0), (800, 576, 4096, 0), (500, 1024, 4096, 0), (100, 768, 8192, 0),
                                               (500, 768, 8192, 0), (800, 512, 16384, 0), (300, 128, 8192, 0), (500, 128, 8192, 0),
                                               (100, 4096, 512, 0), (128, 4096, 512, 0), (64, 8192, 512, 1)])
def test_left_where_it_was(shape, rows, n, k, gated):
    assert shape(rows, n, k, gated) == 0
