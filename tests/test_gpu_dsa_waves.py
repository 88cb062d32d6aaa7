"""Rows of 1 to 16 waves, partly masked, with the row's extremes in any wave: the
range that the waves of a row agree on comes from a reduction over one lane per
wave (quads for rows of up to 4 waves, 16 lanes above), and top_k past the row's
lanes needs several passes of the rank loop.  Integer outputs: exact equality."""
import pytest
import torch

from tests.test_gpu_dsa import case, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("NB,k", [(1024, 1024), (1025, 64), (2048, 600), (3073, 256), (4097, 1024),
                                  (5120, 64), (9217, 512), (15361, 256), (16384, 1024)])
def test_dsa_extremes_in_every_wave(pkg, gpu, dtype, NB, k):
    s, pt, pos, kv = case(NB + k, NB=NB, Q=32, dtype=dtype)
    q = torch.arange(s.shape[2])
    top, low = (q * 509) % NB, (q * 1021 + 7) % NB     # one wave holds each extreme
    s[:, :, q, top] = 37.5
    s[:, :, q, low] = -41.25
    check(pkg, gpu, s, pt, pos, kv, 16, k, f"extremes NB={NB} k={k}")
