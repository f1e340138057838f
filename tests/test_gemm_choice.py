"""Which tiles a product of many rows takes: the host's estimate, asked without a GPU (it then counts 256 CUs)."""
import pytest

from rocml_amd import ops

TILE256, TILE256X192 = 5, 6


# the kind that measured fastest: 256x256 by 8 to 28 % over a choice of smaller tiles, and around them where 256x192 is, by 4 to 15 %
@pytest.mark.parametrize("m,n,k,gated,algo", [
    (384, 24576, 4096, 1, TILE256), (320, 32768, 2048, 1, TILE256), (512, 32768, 2048, 1, TILE256), (257, 32768, 2048, 0, TILE256),
    (129, 151936, 2560, 0, TILE256), (160, 151936, 2560, 0, TILE256), (192, 151936, 4096, 0, TILE256),
    (2643, 4096, 12288, 0, TILE256), (192, 34816, 5120, 0, TILE256X192), (256, 34816, 5120, 1, TILE256X192),
    (512, 19456, 2560, 1, TILE256X192), (1408, 6144, 1024, 1, TILE256X192)])
def test_256_row_tiles(m, n, k, gated, algo):
    assert ops.library("gemm").rocml_gemm_tile_algo(m, n, k, gated) == algo
