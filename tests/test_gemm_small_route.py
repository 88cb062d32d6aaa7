"""The rule that picks a tile for small products (host code only)."""
import pytest

from tests.test_boundary import BASE, fake

SMALL = {(16, 16), (32, 32), (32, 64), (64, 64), (128, 64), (128, 128), (192, 128), (96, 96)}


@pytest.mark.parametrize("M,N,K", [(1, 16, 512), (32, 4096, 7168), (1000, 2112, 7168),
                                   (1500, 4096, 7168), (300, 1024, 2048)])
def test_small_products_take_small_tiles(pkg, M, N, K):
    r = pkg.gemm_route(M, N, K)
    bm, bn = r["block_m"], r["block_n"]
    assert (bm, bn) in SMALL
    assert r["grid_blocks"] == -(-M // bm) * -(-N // bn)
    assert r["block_threads"] == (256 if (bm, bn) in ((64, 64), (96, 96)) else 512)


@pytest.mark.parametrize("M,N,K", [(16384, 4096, 7168), (4096, 4096, 7168),   # one round and more
                                   (5000, 4096, 512),
                                   (32, 4096, 384),              # fewer than 4 k-blocks
                                   (256, 256, 66048 * 128)])     # K past 65536
def test_the_256_row_tiles_stay(pkg, M, N, K):
    r = pkg.gemm_route(M, N, K)
    assert r["block_m"] == 256 and r["block_n"] in (192, 256)


def test_forced_tile_validation(lib):
    def call(block_n, M=0, N=256, K=1024):
        return lib.fagq_gemm_launch_mapped(fake(0), fake(1), fake(2), fake(3), fake(4), M, N, K, 0, 1,
                                           0, block_n, None)
    assert BASE and [call(i) for i in range(9)] == [0] * 9
    assert call(9) == 5 and call(-1) == 5 and call(64) == 5
    assert call(1, K=1 << 17) == 7 and call(1, M=1 << 17) == 7 and call(1, N=1 << 17) == 7
