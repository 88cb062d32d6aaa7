"""The GEMM's tiles for small products against its 256-row tiles and the oracle,
at the sizes where they can go wrong: rows and columns that do not fill a tile,
fewer k-blocks than waves or ring stages, counts that leave the last round of
either ragged, and calls on both sides of the rule that picks a tile.

The ring tiles (64 x 64 and up) sum in k-block order like the 256-row tiles, so
their bits are equal.  The others sum eight interleaved partial sums; any fp32
order stays within the tolerance of test_gpu_gemm.py (see there)."""
import ctypes

import pytest
import torch

from tests.gpu_util import note
from tests.test_gpu_gemm import FORMATS, assert_close, make, run_gpu, run_ref

pytestmark = pytest.mark.gpu

TILES = [(16, 16), (32, 32), (32, 64), (64, 64), (128, 64), (128, 128), (192, 128), (96, 96)]
NAN = float("nan")


def launch(pkg, d, M, N, K, afmt, bfmt, col, block_n):
    c = torch.full((M, N), NAN, dtype=torch.bfloat16, device=d[0].device)
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    st = pkg._lib.load().fagq_gemm_launch_mapped(
        P(d[0]), P(d[1]), P(d[2]), P(d[3]), P(c), M, N, K, 0 if afmt == "f32" else 1,
        1 if col else 0, 0 if bfmt == "f32" else 1, block_n,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == 0, st
    torch.cuda.synchronize()
    return c.cpu()


@pytest.mark.parametrize("afmt,bfmt,col", FORMATS)
@pytest.mark.parametrize("M,N,K", [(1, 16, 512), (17, 144, 128), (33, 208, 640), (65, 80, 1152),
                                   (200, 272, 2176), (193, 400, 384)])
def test_small_tiles_match(pkg, gpu, M, N, K, afmt, bfmt, col):
    note(f"gemm small tiles M={M} N={N} K={K} a={afmt} b={bfmt} col={col}")
    ops = make(M, N, K, afmt, bfmt, col, seed=M + 3 * N + K)
    d = [t.to(gpu).contiguous() for t in ops]
    want = launch(pkg, d, M, N, K, afmt, bfmt, col, 256)
    ref, bound = run_ref(*ops, col)
    for i, (bm, bn) in enumerate(TILES):
        got = launch(pkg, d, M, N, K, afmt, bfmt, col, 1 + i)
        if bm >= 64:
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (bm, bn)
        else:
            assert_close(got.float().numpy(), ref, bound, K, f"{bm}x{bn} of {M}x{N}x{K}")


@pytest.mark.parametrize("nk", [1, 2, 3, 4, 5, 6, 7, 8, 9, 15, 16, 17, 24, 33])
def test_small_tiles_k_block_counts(pkg, gpu, nk):
    # Every remainder of the rings' stages (3, 4 and 5, unrolled 6, 4 and 10
    # times) and of the eight waves, with one and two k-blocks in flight.
    M, N, K = 70, 96, 128 * nk
    note(f"gemm small tiles, {nk} k-blocks")
    for afmt in ("f32", "ue8m0"):
        ops = make(M, N, K, afmt, afmt, True, seed=nk)
        d = [t.to(gpu).contiguous() for t in ops]
        want = launch(pkg, d, M, N, K, afmt, afmt, True, 256)
        ref, bound = run_ref(*ops, True)
        for i, (bm, bn) in enumerate(TILES):
            got = launch(pkg, d, M, N, K, afmt, afmt, True, 1 + i)
            if bm >= 64:
                assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (bm, bn, nk)
            else:
                assert_close(got.float().numpy(), ref, bound, K, f"{bm}x{bn} nk={nk}")


@pytest.mark.parametrize("M,N,K,afmt", [(32, 4096, 1024, "f32"), (5, 640, 4096, "ue8m0"),
                                        (600, 528, 1536, "ue8m0"), (1500, 1040, 512, "f32"),
                                        (2000, 2112, 512, "f32"), (1025, 4608, 512, "ue8m0")])
def test_picked_tile_matches_oracle(pkg, gpu, M, N, K, afmt):
    r = pkg.gemm_route(M, N, K)
    note(f"gemm picked tile {r['block_m']}x{r['block_n']} M={M} N={N} K={K}")
    ops = make(M, N, K, afmt, afmt, True, seed=M)
    got = run_gpu(pkg, gpu, *ops, True)
    rows = torch.arange(0, M, max(1, M // 100))
    ref, bound = run_ref(ops[0][rows], ops[1][:, rows].contiguous(), ops[2], ops[3], True)
    assert_close(got[rows.numpy()], ref, bound, K, f"{M}x{N}x{K}")


def test_infinite_scales_and_special_codes(pkg, gpu):
    # K-blocks past the last read zeros with zero scales: an infinite scale in
    # the real last k-block gives the infinities the 256-row tiles give.
    M, N, K = 20, 48, 640
    note("gemm small tiles, infinite scales")
    a_q, a_s, b_q, b_s = make(M, N, K, "f32", "f32", True, seed=5)
    a_s[-1, 3] = float("inf")
    a_q[7, 5] = NAN
    d = [t.to(gpu).contiguous() for t in (a_q, a_s, b_q, b_s)]
    want = launch(pkg, d, M, N, K, "f32", "f32", True, 256).float()
    assert torch.isinf(want[3]).any() and torch.isnan(want[7]).all()
    for i in range(len(TILES)):
        got = launch(pkg, d, M, N, K, "f32", "f32", True, 1 + i).float()
        assert torch.equal(torch.isnan(got), torch.isnan(want)), TILES[i]
        assert torch.equal(torch.isinf(got), torch.isinf(want)), TILES[i]


@pytest.mark.parametrize("afmt,bfmt,col", FORMATS)
@pytest.mark.parametrize("M,N", [(97, 400), (95, 1104), (192, 96), (50, 208)])
def test_96_column_tiles_straddle_weight_blocks(pkg, gpu, M, N, afmt, bfmt, col):
    # Tiles from columns 96, 192, 288 and 384: their waves of 48 columns meet the
    # 128-column boundaries after 0 to 3 of their 16-column tiles; N ends a tile
    # inside a wave, in its first block and past its last.
    K = 896
    note(f"gemm 96 x 96 tile M={M} N={N} a={afmt} b={bfmt} col={col}")
    ops = make(M, N, K, afmt, bfmt, col, seed=M + N)
    d = [t.to(gpu).contiguous() for t in ops]
    want = launch(pkg, d, M, N, K, afmt, bfmt, col, 256)
    got = launch(pkg, d, M, N, K, afmt, bfmt, col, 1 + TILES.index((96, 96)))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
