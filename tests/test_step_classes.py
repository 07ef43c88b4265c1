"""Recorded steps are padded to the rows of their size class: a product's kernel, and with it the order of its additions,
must be the class's for every step of the class, so that a step adds the same way recorded and not."""
import ctypes

import pytest

from minivllm_amd.engine.executor import GRAPH_BUCKETS, TOKEN_BUCKETS


@pytest.fixture(scope="module")
def served():
    from minivllm_amd.csrc import build
    path = build.find_library("bf16") or build.build("bf16")
    shape = ctypes.CDLL(path).mv_gemm_deep_shape
    return lambda rows, n, k, gated: shape(rows, n, k, gated) != 0


# weights of the 0.6B and 8B sizes, and others whose tiles fill the units at other numbers of rows
@pytest.mark.parametrize("n,k,gated", [(4096, 1024, 0), (6144, 1024, 1), (1024, 2048, 0), (1024, 3072, 0), (6144, 4096, 0), (4096, 4096, 0),
                                       (4096, 12288, 0), (24576, 4096, 1), (1792, 1024, 0), (1152, 1024, 0), (512, 2048, 0), (768, 1536, 0),
                                       (3584, 768, 1), (640, 2048, 0), (64, 1024, 0)])
@pytest.mark.parametrize("kind", ["decode", "prompt"])
def test_a_class_has_one_product(served, n, k, gated, kind):
    classes = GRAPH_BUCKETS if kind == "decode" else TOKEN_BUCKETS
    for rows in range(1, min(classes[-1], 1200) + 1):
        padded = next(b for b in classes if b >= rows)
        assert served(rows, n, k, gated) == served(padded, n, k, gated), (rows, padded)
