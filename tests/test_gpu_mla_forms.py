"""The MLA backward's long form (whole rows per workgroup, three launches) and its
head planes (the heads halved over workgroups), at the sizes where they can go
wrong: column slices, alone and beside a short slice over the same workspace;
widths whose lanes do not divide a workgroup; the narrowest ones; odd numbers of
heads to halve, with both numbers of heads in flight; sequences that end inside a
block of 8 or 16 rows.  Each case
states the form it means to run.  Oracle and bars: test_gpu_mla.py."""
import random

import pytest
import torch

from tests.test_gpu_mla import case

pytestmark = pytest.mark.gpu

F32, BF16 = torch.float32, torch.bfloat16


def forms(B, H, S, D, grad):
    """(dims of a tile or 0, heads in flight, head planes) of each column slice."""
    from fagq_mi355x import _lib
    rs = [_lib.query_mla_route(B, H, S, D, grad == F32, sl) for sl in range(-(-D // 512))]
    return [(r["tile_dims"], r["heads_in_flight"], r["head_planes"]) for r in rs]


@pytest.mark.parametrize("B,H,S,D,grad,want", [
    (1, 3, 4100, 576, BF16, [(0, 2, 1), (64, 4, 1)]),       # long, then short
    (1, 2, 2050, 576, F32, [(0, 1, 1), (64, 4, 1)]),
    (1, 2, 4100, 1024, BF16, [(0, 2, 1), (0, 2, 1)]),       # long twice
    (1, 3, 2050, 1024, F32, [(0, 1, 1), (0, 1, 1)]),
])
def test_long_column_slices(pkg, gpu, B, H, S, D, grad, want):
    assert forms(B, H, S, D, grad) == want
    case(pkg, gpu, B, H, S, D, grad, seed=D + S)


@pytest.mark.parametrize("B,H,S,D,grad,want", [
    (1, 2, 5111, 192, F32, (0, 1, 1)), (2, 3, 1537, 320, F32, (0, 1, 1)),
    (1, 1, 2049, 448, F32, (0, 1, 1)), (8, 1, 2049, 64, F32, (0, 1, 1)),
    (4, 2, 2049, 128, F32, (0, 1, 1)), (16, 2, 2049, 64, BF16, (0, 2, 1)),
    (8, 3, 2049, 128, BF16, (0, 2, 1)), (2, 2, 5201, 192, BF16, (0, 2, 1)),
    (1, 2, 6000, 192, BF16, (0, 8, 1)), (1, 9, 3001, 448, BF16, (0, 8, 1)),
    (1, 3, 4096, 512, BF16, (0, 8, 1)), (3, 5, 1367, 512, BF16, (0, 2, 1)),
])
def test_long_widths(pkg, gpu, B, H, S, D, grad, want):
    assert forms(B, H, S, D, grad) == [want]
    case(pkg, gpu, B, H, S, D, grad, seed=S)


@pytest.mark.parametrize("B,H,S,D,grad,want", [
    (1, 65, 1285, 512, F32, (0, 1, 2)), (2, 49, 1283, 256, F32, (0, 1, 2)),
    (1, 67, 2077, 512, BF16, (0, 2, 2)), (1, 64, 4161, 256, BF16, (0, 2, 2)),
])
def test_long_head_planes(pkg, gpu, B, H, S, D, grad, want):
    assert forms(B, H, S, D, grad) == [want]
    case(pkg, gpu, B, H, S, D, grad, seed=S)


@pytest.mark.parametrize("B,H,S,D,want", [
    (1, 40, 1, 64, (64, 4, 2)), (2, 49, 37, 192, (64, 4, 2)), (1, 129, 17, 512, (64, 4, 2)),
    (1, 48, 1024, 64, (64, 4, 2)), (1, 51, 79, 448, (64, 4, 2)), (1, 113, 230, 448, (64, 4, 2)),
    (1, 128, 150, 512, (128, 8, 2)), (1, 50, 1021, 128, (128, 4, 2)), (1, 65, 255, 512, (128, 4, 2)),
    (2, 53, 165, 384, (128, 4, 2)), (1, 129, 421, 512, (128, 8, 2)), (2, 65, 299, 512, (128, 4, 2)),
    (3, 65, 427, 512, (128, 8, 2)), (3, 41, 342, 384, (128, 8, 2)), (3, 64, 1333, 256, (128, 8, 1)),
    (1, 64, 100, 640, (128, 4, 2)),
])
@pytest.mark.parametrize("grad", [F32, BF16])
def test_short_head_planes(pkg, gpu, B, H, S, D, want, grad):
    got = forms(B, H, S, D, grad)
    assert got[0] == want
    case(pkg, gpu, B, H, S, D, grad, seed=S + H)


@pytest.mark.parametrize("seed", range(12))
def test_random_long(pkg, gpu, seed):
    rng = random.Random(7000 + seed)
    grad = rng.choice([F32, BF16])
    D = 64 * rng.randint(1, 10)
    rows = 256 // (min(D, 512) // 8)                        # of a workgroup of the first slice
    B, H = rng.randint(1, 4), rng.randint(1, 3)
    S = rows * -(-(512 if grad == F32 else 1024) // B) + rng.randint(0, 2 * rows)
    assert forms(B, H, S, D, grad)[0][0] == 0
    case(pkg, gpu, B, H, S, D, grad, rng.choice([None, F32, BF16]), seed=seed)


@pytest.mark.parametrize("B,H,S,D,grad", [(1, 128, 34, 512, F32), (1, 128, 150, 512, BF16), (1, 4, 40, 576, F32),
                                          (1, 48, 1024, 64, BF16), (1, 48, 1283, 512, F32), (1, 3, 4096, 512, BF16),
                                          (1, 3, 4100, 576, BF16), (2, 49, 37, 192, F32)])
def test_workspace_of_the_told_size(pkg, gpu, B, H, S, D, grad):
    """No form writes past the workspace bytes that a caller is told, and its results do
    not depend on what they held."""
    from fagq_mi355x import mla_bwd
    from fagq_mi355x.workloads import MlaWorkload, make_mla_inputs
    from tests.gpu_util import note
    note(f"mla workspace B{B} H{H} S{S} D{D} {grad}")
    w = MlaWorkload("t", B, H, S, D, grad, seed=S)
    q, c, out, do, lse = make_mla_inputs(w, device=gpu)
    need = mla_bwd.workspace_bytes(B, S, D)
    got = []
    for fill in (0, 0xFF):                                  # 0xFF: NaN as fp32
        buf = torch.full((need + 8192,), 0xA5, dtype=torch.uint8, device=gpu)
        buf[:need] = fill
        dq, dc = torch.empty_like(q, dtype=grad), torch.empty_like(c, dtype=grad)
        pkg.mla_bwd_nope_dkdv(q, c, out, do, lse, dq, dc, w.sm_scale, workspace=buf[:need])
        torch.cuda.synchronize()
        assert bool((buf[need:] == 0xA5).all())
        got.append((dq, dc))
    for a, b in zip(*got):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
