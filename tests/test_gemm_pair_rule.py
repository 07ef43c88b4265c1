"""Which gated pairs the product for prompts takes, and its tiles: sizes at which all sides were measured."""
import ctypes

import pytest

from minivllm_amd.engine.executor import GRAPH_BUCKETS, TOKEN_BUCKETS


@pytest.fixture(scope="module")
def lib():
    from minivllm_amd.csrc import build
    return ctypes.CDLL(build.find_library("bf16") or build.build("bf16"))


@pytest.fixture(scope="module")
def shape(lib):
    return lib.mv_gemm_pair_shape


@pytest.mark.parametrize("rows, n, k, bm, bn", [(320, 6144, 1024, 64, 128), (640, 6144, 1024, 128, 128), (1024, 6144, 1024, 128, 192),
                                                (1280, 6144, 1024, 256, 128), (1536, 6144, 1024, 192, 192), (2048, 6144, 1024, 256, 192),
                                                (1024, 12288, 2048, 256, 192), (512, 1536, 512, 64, 64)])
def test_served(shape, rows, n, k, bm, bn):
    assert divmod(shape(rows, n, k, 256), 1 << 16) == (bm, bn)


@pytest.mark.parametrize("rows, n, k", [(96, 6144, 1024), (128, 6144, 1024), (200, 24576, 4096), (800, 24576, 4096), (4415, 24576, 4096), (8192, 6144, 1024),
                                        (4096, 12288, 2048), (300, 51200, 5120), (300, 6145, 1024), (300, 6144, 1000)])
def test_left_where_it_was(shape, rows, n, k):
    assert shape(rows, n, k, 256) == 0


@pytest.mark.parametrize("n, k", [(6144, 1024), (1536, 1024), (5632, 1024), (8192, 1024), (3072, 1024), (5632, 2048), (12288, 2048), (19456, 2560),
                                  (24576, 4096)])
@pytest.mark.parametrize("classes", [GRAPH_BUCKETS, TOKEN_BUCKETS], ids=["decode", "prompt"])
def test_a_class_has_one_product(shape, n, k, classes):
    """What serves instead rounds elsewhere, so a step of a size class must take the same one recorded (padded to the class) and not."""
    for rows in range(129, classes[-1] + 1):
        padded = next(b for b in classes if b >= rows)
        assert bool(shape(rows, n, k, 256)) == bool(shape(padded, n, k, 256)), (rows, padded)


@pytest.mark.parametrize("rows, n, k, bm, bn", [(224, 3104, 1024, 64, 64), (576, 1024, 1024, 64, 64), (1024, 3104, 1024, 128, 128),
                                                (2048, 5184, 1024, 256, 192), (2048, 4112, 1024, 192, 192), (1024, 3072, 256, 128, 96)])
def test_plain_products_served(lib, rows, n, k, bm, bn):
    assert divmod(lib.mv_gemm_round_shape(rows, n, k, 256), 1 << 16) == (bm, bn)


# one request's and few rows, long K, full tiles of the library's, more than a round; what gemm_deep.hip takes
@pytest.mark.parametrize("rows, n, k", [(128, 5184, 1024), (2048, 1024, 3072), (2048, 1024, 2048), (2048, 4096, 1024), (4096, 3104, 1024), (4415, 24576, 4096),
                                        (512, 1024, 2048), (160, 1040, 1024), (300, 5184, 1000), (1024, 151936, 1024)])
def test_plain_products_left_where_they_were(lib, rows, n, k):
    assert lib.mv_gemm_round_shape(rows, n, k, 256) == 0


@pytest.mark.parametrize("n, k", [(5184, 1024), (3104, 1024), (1024, 1024), (592, 1024), (2080, 512), (6176, 2048), (3072, 256), (1024, 2048)])
@pytest.mark.parametrize("classes", [GRAPH_BUCKETS, TOKEN_BUCKETS], ids=["decode", "prompt"])
def test_a_class_has_one_plain_product(lib, n, k, classes):
    shape = lib.mv_gemm_round_shape
    for rows in range(129, classes[-1] + 1):
        padded = next(b for b in classes if b >= rows)
        assert bool(shape(rows, n, k, 256)) == bool(shape(padded, n, k, 256)), (rows, padded)


@pytest.mark.parametrize("rows, n, k, here", [(4096, 4096, 2048, False), (5120, 6144, 1024, False), (4096, 8192, 1024, False), (4096, 6144, 1024, True),
                                              (2560, 6144, 1024, True), (2048, 8192, 1024, True), (5784, 4896, 768, True), (1655, 10528, 1024, True)])
def test_a_weight_of_the_librarys_tiles_has_to_be_ahead(shape, rows, n, k, here):
    assert (shape(rows, n, k, 256) != 0) is here


@pytest.mark.parametrize("M, N, K", [(1024, 6144, 1024), (64, 6144, 1024)])
def test_a_pair_with_a_squared_relu_stays_refused(lib, M, N, K):
    """Whichever kernel would take the pair: none of them squares it. (Refused in front of any launch: the addresses are made up.)"""
    lib.mv_last_error.restype = ctypes.c_char_p
    p, i, n, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_long, ctypes.c_float
    lib.mv_gemm_tile.argtypes = [p, n, p, p, p, n, i, i, i, i, i, p, n, i, f, f, i, p]
    address, bf16 = 1 << 20, 1
    assert lib.mv_gemm_tile(address, K, address, None, address, N // 2, bf16, M, N, K, 1, None, 0, 0, 0.0, 1.0, 1, None)
    assert b"squared ReLU" in lib.mv_last_error()


@pytest.mark.parametrize("lda, n, k, reaches", [(1024, 6144, 1024, 1), ((1 << 23) - 8, 6144, 1024, 1), (1 << 23, 6144, 1024, 0), (1 << 40, 64, 64, 0),
                                                (4096, (1 << 19) - 1, 4096, 1), (4096, 1 << 19, 4096, 0)])
def test_offsets_of_a_tile_fit_into_32_bits(lib, lda, n, k, reaches):
    """A lane's byte offset is at most that of row 255 of a tile, or of the weight's last row, and a chunk's 128 bytes."""
    lib.mv_gemm_pair_reaches.argtypes = [ctypes.c_long, ctypes.c_int, ctypes.c_int]
    assert lib.mv_gemm_pair_reaches(lda, n, k) == reaches
    assert not reaches or max(255 * lda, (n - 1) * k) * 2 + 128 < 1 << 32


@pytest.mark.parametrize("n, k, gated", [(1024, 2048, None), (1024, 3072, None), (384, 64, None), (2048, 1024, None), (6144, 1024, 1), (2048, 1024, 1), (4096, 1024, 0),
                                         (5184, 1024, 0), (592, 1024, 0)])
@pytest.mark.parametrize("classes", [GRAPH_BUCKETS, TOKEN_BUCKETS], ids=["decode", "prompt"])
def test_a_class_has_one_way_through_a_norm(lib, n, k, gated, classes):
    serves = (lambda m: lib.mv_gemm_into_norm_parts(m, n, k, 256)) if gated is None else lambda m: lib.mv_gemm_behind_norm_serves(m, n, k, gated, 256)
    for rows in range(97, min(classes[-1], 1200) + 1):
        assert serves(rows) == serves(next(b for b in classes if b >= rows)), rows


def test_sizes_whose_norm_stays_apart(lib):
    assert all(lib.mv_gemm_into_norm_parts(m, n, k, 256) == 0 for m, n, k in [(128, 1024, 2048), (1025, 1024, 2048), (300, 4096, 4096), (300, 1088, 2048), (300, 1024, 2000)])
    assert all(lib.mv_gemm_behind_norm_serves(*a, 256) == 0 for a in [(128, 4096, 1024, 0), (1025, 4096, 1024, 0), (600, 24576, 4096, 1), (1024, 20480, 1024, 0), (300, 6145, 1024, 1)])
