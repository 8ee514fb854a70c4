"""Which weight gradients in 16 bits are this package's own, and how much scratch they take."""
import ctypes

import pytest

from quick_ssm_amd import _lib


# us measured for the library's product and this package's, bf16
@pytest.mark.parametrize("rows,n,k,library,own", [
    (8192, 128, 128, 62, 22), (8192, 5120, 1024, 117, 88), (16384, 1024, 4096, 174, 131), (12288, 5120, 1280, 284, 155),
    (8192, 12800, 512, 116, 127), (8192, 10240, 1024, 162, 191), (12288, 10240, 1024, 248, 294), (12288, 11520, 1024, 270, 303),
    (16384, 11520, 1024, 352, 442), (16384, 3072, 3072, 284, 308), (16384, 12800, 640, 276, 360), (8192, 12800, 1024, 276, 185),
    (8192, 16384, 1024, 230, 219), (8192, 17920, 1024, 319, 264), (16384, 20480, 1024, 868, 683), (8192, 8, 8, 13, 22),
    (8192, 48, 48, 16, 22), (16384, 512, 8, 28, 29), (24576, 8, 8, 31, 28), (4096, 10240, 1024, 88, 100), (2048, 1024, 1024, 20, 28),
])
def test_the_faster_product_is_taken(rows, n, k, library, own):
    assert bool(_lib.load().qssm_weight_gradient_suits(n, k, rows)) == (own < library)


def test_scratch_is_bounded():
    lib = _lib.load()
    lib.qssm_weight_gradient_floats.restype = ctypes.c_uint64
    for rows in (64, 8192, 1 << 17, 1 << 20, (1 << 30) - 8):
        for n in (8, 256, 2816, 10240, 20480):
            for k in (8, 1024, 2816, 4096):
                # two rounds of parts of a tile each
                assert lib.qssm_weight_gradient_floats(n, k, rows) <= 512 * 256 * 256
