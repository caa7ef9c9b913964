"""Which kernel an FP8 GEMM takes, on the CPU (the planner assumes the card's
256 CUs where there is none)."""
import random

import pytest

BIAS, ROWMAX, GATE = 0, 1, 2


def _tile(M, N, K, epi, rows16=1):
    from flashvsr_sm89_ops import _lib
    return _lib.lib().fvsr_gemm_tile(M, N, K, epi, rows16).decode()


# Measured on an MI355X (us): the kernel named is the fastest or within 3% of
# it; beside it what a choice by K steps alone took, 9% to 40% more.
@pytest.mark.parametrize("M,N,K,epi,rows16,want", [
    (12300, 1400, 1536, BIAS, 1, ("64x128",)),              # 42.1; 128x128 52.3
    (14500, 1400, 1536, BIAS, 1, ("64x128", "ring")),       # 47.0, 48.8; 128x128 54.3
    (4224, 4600, 1536, BIAS, 1, ("64x128", "ring")),        # 45.9, 47.9; 128x128 52.3
    (12300, 1536, 1536, BIAS, 0, ("64x128", "ring")),       # 56.5, 57.4; 128x128 62.5
    (2304, 8960, 1536, BIAS, 0, ("64x128", "ring")),        # 56.2, 58.9; 128x128 62.5
    (5014, 1280, 4096, ROWMAX, 1, ("ring128",)),            # 30.8; 128x256 34.5
    (16896, 1280, 4096, BIAS, 1, ("ring192",)),             # 72.4; 128x256 93.2
    (12300, 1536, 8960, BIAS, 1, ("ring192",)),             # 137.8; 128x256 158.2
    (7000, 1400, 1536, GATE, 1, ("64x128",)),               # 30.6; ring 42.8
    (12300, 1536, 1536, GATE, 1, ("64x128",)),              # 53.1; 128x128 69.3
    (2079, 4600, 1536, ROWMAX, 1, ("64x128",)),             # 27.8; ring 34.6
    # ... and lines that stay where they were
    (512, 1536, 1536, BIAS, 1, ("64x64",)), (2079, 1536, 1536, BIAS, 1, ("128x128",)),
    (1152, 1536, 8960, BIAS, 1, ("64x128",)), (4224, 1536, 1536, BIAS, 1, ("ring128",)),
    (8448, 8960, 1536, ROWMAX, 1, ("ring256",)), (16896, 4608, 1536, BIAS, 1, ("ring256",)),
    (16896, 1536, 8960, BIAS, 1, ("ring256 prefetching",)),
])
def test_measured_choices(M, N, K, epi, rows16, want):
    assert _tile(M, N, K, epi, rows16) in want


def test_kernels_only_where_they_apply():
    rng = random.Random(0)
    seen = set()
    for _ in range(4000):
        M, N = (int(2 ** rng.uniform(0, 15)) for _ in range(2))
        N = rng.choice((N, -(-N // 256) * 256))
        K = rng.choice((16, 48, 128, 256, 384, 512, 768, 1024, 1536, 1664, 4096, 4224, 8960))
        epi, rows16 = rng.randrange(3), rng.randrange(2)
        t = _tile(M, N, K, epi, rows16)
        seen.add(t)
        assert (t == "generic") == (K % 128 != 0)
        if t.startswith("ring"):
            assert K % 256 == 0 and K >= 512
            assert (t == "ring") == (epi == GATE or not rows16 or N % 256 != 0)
        assert t != "64x64" or epi != ROWMAX
        assert t != "ring256" or K < 4096
    assert seen == {"generic", "64x64", "64x128", "128x128", "128x256", "ring", "ring128",
                    "ring192", "ring256", "ring256 prefetching"}
    for bad in ((0, 8, 128, 0), (8, 0, 128, 0), (8, 8, 0, 0), (8, 8, 128, 3), (8, 8, 128, -1)):
        assert _tile(*bad) == ""


def test_shapes_of_the_gpu_tests_reach_every_kernel():
    """The GPU tests' shapes run every kernel with each epilogue it has, on a
    ragged last row tile, on a ragged last column tile where it takes one, and at
    every remainder of the small tiles' trips."""
    from test_gpu_gemm_tiles import _SHAPES
    size = {"64x64": (64, 64, 4), "64x128": (64, 128, 6), "128x128": (128, 128, 4),
            "128x256": (128, 256, 6), "ring": (256, 256, 1), "ring128": (128, 256, 1),
            "ring192": (192, 256, 1), "ring256": (256, 256, 1),
            "ring256 prefetching": (256, 256, 1)}
    for epi in (BIAS, ROWMAX, GATE):
        reached = {}
        for shape in _SHAPES:
            reached.setdefault(_tile(*shape, epi), []).append(shape)
        want = set(size) - {"64x64"} if epi == ROWMAX else set(size)
        if epi == GATE:
            want -= {"ring128", "ring192", "ring256", "ring256 prefetching"}
        assert set(reached) == want
        for t, shapes in reached.items():
            rows, cols, trip = size[t]
            assert any(M % rows for M, _, _ in shapes)
            assert any(N % cols for _, N, _ in shapes) or t[:5] in ("ring1", "ring2")
            assert {K // 128 % trip for _, _, K in shapes} == set(range(trip)), (t, epi)
