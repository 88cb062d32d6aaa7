"""The MLA backward's short-sequence kernels at the sizes where they can go wrong:
sequences that do not fill a block of 8 rows or a scan block, every column tile
(dims 64, 128, 256 and 512 wide, with 8 to 1 head groups and fewer heads than
groups), column slices, and both sides of the lines between the tiles and
between short and long sequences.  Oracle and bars: test_gpu_mla.py."""
import pytest
import torch

from tests.test_gpu_mla import case

pytestmark = pytest.mark.gpu

F32, BF16 = torch.float32, torch.bfloat16


@pytest.mark.parametrize("B,H,S,D", [(1, 2, 7, 64), (1, 3, 8, 128), (2, 2, 9, 192), (1, 1, 65, 576),
                                     (3, 9, 129, 512), (2, 40, 136, 512), (1, 3, 1287, 256)])
@pytest.mark.parametrize("grad", [F32, BF16])
def test_short_blocks_and_tiles(pkg, gpu, B, H, S, D, grad):
    case(pkg, gpu, B, H, S, D, grad, seed=S)


@pytest.mark.parametrize("S,grad", [(2552, BF16), (2553, BF16),      # 319 and 320 workgroups of 512 dims
                                    (1276, F32), (1281, F32),        # 256 dims: 320 and 322
                                    (4092, BF16), (4093, BF16),      # the last short sequence, long
                                    (2044, F32), (2045, F32)])       # the same with fp32 dq
def test_lines_between_tiles(pkg, gpu, S, grad):
    case(pkg, gpu, 1, 2, S, 512, grad, seed=S)


@pytest.mark.parametrize("S", [1712, 1721])                          # 1498 and 1512 workgroups of 64 dims
def test_line_of_64_dim_tiles(pkg, gpu, S):
    case(pkg, gpu, 1, 3, S, 448, BF16, seed=S)
