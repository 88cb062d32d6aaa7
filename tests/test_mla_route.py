"""The rule that picks the MLA backward's form and tile (host code only)."""
import pytest


def route(B, H, S, D, f32, slice=0):
    from fagq_mi355x import _lib
    r = _lib.query_mla_route(B, H, S, D, f32, slice)
    return r["tile_dims"], r["heads_in_flight"], r["head_planes"]


LONG2, LONG1, LONG8 = (0, 2, 1), (0, 1, 1), (0, 8, 1)


@pytest.mark.parametrize("B,H,S,D,f32,want", [
    # the long form: one round of 4 workgroups per CU, and both sides of it
    (2, 64, 2048, 512, False, LONG8), (2, 64, 2040, 512, False, (512, 4, 1)),
    (2, 64, 2052, 512, False, LONG2), (1, 2, 4092, 512, False, (512, 4, 1)),
    (1, 2, 2044, 512, True, (256, 4, 1)), (1, 2, 2045, 512, True, LONG1),
    # widths that only 64-dim tiles fit, few heads
    (1, 8, 3000, 448, False, LONG8), (1, 16, 3000, 448, False, (64, 4, 1)),
    (1, 8, 1700, 448, False, (64, 4, 1)),
    # the widest tile of 320 workgroups, else 128 dims beside the exact rows, else 64
    (2, 64, 1900, 512, False, (512, 4, 1)), (2, 64, 1024, 512, False, (256, 4, 1)),
    (1, 8, 769, 512, False, (128, 4, 1)), (4, 24, 100, 512, True, (128, 8, 1)),
    (8, 24, 100, 512, True, (128, 4, 1)), (8, 24, 60, 512, True, (64, 4, 1)),
    (1, 16, 40, 320, False, (64, 4, 1)), (1, 64, 300, 512, True, (128, 8, 1)),
    # 40 heads and more, halved: at most one 128-dim tile per CU ..
    (1, 128, 34, 512, True, (64, 4, 2)), (1, 128, 97, 512, True, (128, 8, 2)),
    (1, 128, 256, 512, False, (128, 8, 2)), (1, 111, 256, 512, False, (128, 4, 2)),
    (1, 64, 256, 512, True, (128, 4, 2)), (1, 64, 257, 512, True, (128, 8, 1)),
    (3, 128, 32, 512, True, (64, 4, 2)), (3, 128, 33, 512, True, (128, 4, 2)),
    (1, 40, 34, 512, True, (64, 4, 2)), (1, 39, 34, 512, True, (128, 8, 1)),
    (1, 48, 1024, 128, False, (128, 4, 2)), (1, 48, 1025, 128, False, (128, 8, 1)),
    # .. or where the tiles do not fit one round with the exact rows
    (1, 128, 420, 512, True, (128, 8, 2)), (2, 64, 300, 512, False, (128, 4, 2)),
    (1, 64, 632, 512, True, (128, 4, 2)), (1, 64, 633, 512, True, (128, 4, 1)),
    (8, 64, 31, 512, False, (128, 4, 2)),
    (8, 65, 31, 512, False, (64, 4, 1)), (8, 65, 32, 512, False, (128, 4, 2)),
    # .. odd widths
    (1, 64, 145, 448, False, (64, 4, 1)), (1, 64, 144, 448, False, (64, 4, 2)),
    (2, 64, 31, 448, False, (64, 4, 1)), (1, 64, 31, 448, False, (64, 4, 2)),
    (2, 112, 224, 448, True, (64, 4, 2)), (2, 112, 233, 448, True, (64, 4, 1)),
    (2, 111, 224, 448, True, (64, 4, 1)),
    # .. three batches
    (3, 64, 424, 512, True, (128, 8, 2)), (4, 40, 255, 384, False, (128, 8, 2)),
    (2, 128, 457, 512, False, (128, 4, 1)), (4, 64, 850, 512, False, (128, 8, 2)),
    (3, 64, 1333, 256, False, (128, 8, 1)), (4, 63, 850, 512, False, (512, 4, 1)),
    # .. whole rows instead of tiles
    (1, 128, 1300, 512, True, (0, 1, 2)), (1, 47, 1300, 512, True, (256, 4, 1)),
    (1, 48, 1536, 512, True, (0, 1, 2)), (1, 48, 1537, 512, True, (256, 4, 1)),
    (2, 64, 640, 512, True, (0, 1, 2)), (2, 64, 632, 512, True, (128, 4, 1)),
    (1, 64, 2073, 512, False, (0, 2, 2)), (1, 64, 2072, 512, False, (256, 4, 1)),
    (1, 128, 3032, 512, False, (0, 2, 2)), (1, 128, 3033, 512, False, (512, 4, 1)),
    (2, 128, 1272, 512, False, (0, 2, 2)), (2, 128, 1273, 512, False, (512, 4, 1)),
    (2, 95, 1272, 512, False, (256, 4, 1)), (1, 63, 2400, 512, False, (256, 4, 1)), (1, 64, 4160, 256, False, (0, 2, 2)),
    (1, 128, 2400, 384, False, (128, 4, 1)),
])
def test_form(pkg, B, H, S, D, f32, want):
    assert route(B, H, S, D, f32) == want


def test_slices_pick_their_own_form(pkg):
    assert route(1, 3, 4100, 576, False, 0) == LONG2 and route(1, 3, 4100, 576, False, 1) == (64, 4, 1)
    assert route(1, 3, 4100, 1024, False, 0) == route(1, 3, 4100, 1024, False, 1) == LONG2


def test_query_errors(pkg, lib):
    import ctypes
    from fagq_mi355x import _lib
    r = _lib.MlaRoute()
    q = lambda *a: lib.fagq_mla_bwd_query_route(*a, ctypes.byref(r))
    assert q(1, 2, 3, 64, 1, 0) == 0 and r.dims == 64
    assert q(0, 2, 3, 64, 1, 0) == 0
    assert q(1, 2, 3, 64, 2, 0) == 5                      # dq_dtype
    for a in ((-1, 2, 3, 64, 1, 0), (1, 0, 3, 64, 1, 0), (1, 2, 0, 64, 1, 0), (1, 2, 3, 96, 1, 0),
              (1, 2, 3, 64, 1, 1), (1, 2, 3, 64, 1, -1), (1, 2, 3, 576, 1, 2)):
        assert q(*a) == 2, a
    assert q(65536, 2, 3, 64, 1, 0) == 7 and q(1, 64, 1 << 20, 64, 1, 0) == 7
    assert lib.fagq_mla_bwd_query_route(1, 2, 3, 64, 1, 0, None) == 1


def test_the_workspace_holds_what_a_form_uses(pkg, lib):
    """Every slice's planes of head sums and block totals fit the size a caller is told."""
    import random
    from fagq_mi355x import _lib
    rng = random.Random(3)
    for _ in range(4000):
        B, H, D = rng.randint(1, 9), rng.choice((1, 8, 39, 40, 48, 64, 128)), 64 * rng.randint(1, 20)
        S, f32 = int(2 ** rng.uniform(0, 13.5)), rng.random() < 0.5
        if H * S * D * 4 >= 1 << 32:
            continue
        rows = min(max((-(-S // 64) + 15) // 16 * 16, 16), 64)
        need = lib.fagq_mla_bwd_workspace_bytes(B, S, D)
        for sl in range(-(-D // 512)):
            r = _lib.query_mla_route(B, H, S, D, f32, sl)
            assert r["dims"] == min(512, D - 512 * sl)
            totals = 0 if r["tile_dims"] else B * -(-S // rows)
            assert need >= (r["head_planes"] * B * S + totals) * r["dims"] * 4, (B, H, S, D, f32, sl)
            if r["tile_dims"] and r["head_planes"] == 2:
                assert rows == 16 and H >= 40             # the two-plane scan's registers
