"""The tiles of a mixture's products over chosen pairs: those that were measured fastest, or near it."""
import ctypes

import pytest

from minivllm_amd.csrc import build as kernel_build


@pytest.mark.parametrize("n, E, top, hid, F, FS, rows, columns, down", [
    (8, 32, 4, 1024, 768, 0, 32, 128, 128), (1, 32, 4, 1024, 768, 0, 32, 64, 64), (100, 32, 4, 1024, 768, 768, 32, 256, 256),
    (100, 32, 4, 1024, 768, 0, 32, 256, 128), (256, 32, 4, 1024, 768, 768, 64, 256, 256), (512, 32, 4, 1024, 768, 768, 96, 256, 256),
    (768, 32, 4, 1024, 768, 768, 128, 256, 256), (1000, 32, 4, 1024, 768, 768, 160, 256, 256), (1500, 32, 4, 1024, 768, 768, 128, 256, 256),
    (2048, 32, 4, 1024, 768, 0, 160, 256, 256), (200, 16, 4, 1024, 768, 768, 64, 128, 128), (1000, 8, 2, 4096, 3072, 0, 160, 256, 256)])
def test_tiles_of_measured_mixtures(n, E, top, hid, F, FS, rows, columns, down):
    lib = kernel_build.find_library("bf16") or kernel_build.build("bf16")
    shape = ctypes.CDLL(lib).mv_moe_pairs_shape(n, top, E, hid, F, FS, 256)
    assert (shape & 1023, shape >> 10 & 1023, shape >> 20) == (rows, columns, down)


@pytest.mark.parametrize("n, E, top, hid, F, FS, rows, columns, down", [
    (8, 64, 8, 2048, 768, 0, 32, 128, 128), (128, 64, 8, 2048, 768, 0, 32, 128, 128), (256, 64, 8, 2048, 768, 0, 64, 128, 128),
    (33, 128, 8, 1024, 384, 0, 32, 128, 128), (8, 128, 8, 1024, 384, 0, 32, 256, 256), (33, 16, 2, 4096, 1536, 0, 32, 128, 128),
    (400, 16, 2, 4096, 1536, 0, 64, 128, 128), (600, 16, 2, 4096, 1536, 0, 96, 256, 256)])
def test_low_tiles_are_wide_in_one_short_round_only(n, E, top, hid, F, FS, rows, columns, down):
    test_tiles_of_measured_mixtures(n, E, top, hid, F, FS, rows, columns, down)
