"""Which sparse attention calls run some units as several workgroups, on the
CPU (the planner assumes the card's 256 CUs where there is none)."""
import pytest

PIECE = 128 * 128 + 2 * 128  # floats of one piece's partial result


def _pieces(H, NQ, maxk):
    from flashvsr_sm89_ops import _lib
    n = _lib.lib().fvsr_bsa_workspace_floats(H, NQ, maxk)
    units = H * NQ
    rest = units % 256
    assert n == 0 or (rest and n % (rest * PIECE) == 0)
    return n // (rest * PIECE) if n else 1


# Measured on an MI355X (us, whole / in two or three pieces each): the pieces'
# partial results and second launch cost more than the blocks they save.
@pytest.mark.parametrize("H,NQ,maxk", [
    (12, 8, 8),     # every block kept: 24.8 / 26.3 at 96 units
    (12, 9, 9),     # 24.8 / 27.0 ; a fifth kept 18.1 / 19.9
    (12, 11, 11),   # a fifth kept 21% slower, all 19%
    (12, 13, 13),   # a fifth 16%, all 4%
    (8, 25, 25),    # a fifth 11%
    (12, 20, 20),   # a fifth 27%, all 8%
    (12, 36, 36),   # 139.7 / 148.9
    (12, 36, 144),  # 514.8 / 545.9
])
def test_not_split(H, NQ, maxk):
    assert _pieces(H, NQ, maxk) == 1


@pytest.mark.parametrize("H,NQ,maxk,want", [
    (1, 1, 8, 2), (1, 2, 16, 4), (4, 4, 8, 2), (8, 4, 8, 2), (8, 10, 10, 2), (12, 4, 16, 4), (12, 9, 18, 4),
    (12, 9, 36, 4), (4, 9, 36, 8), (12, 17, 68, 2), (12, 21, 63, 2), (4, 36, 72, 3),
    # past a multiple of the CUs: at least 8 entries of the index row to a piece, at most 4
    (12, 23, 23, 2), (12, 24, 24, 3), (12, 66, 66, 4), (12, 66, 198, 4), (12, 55, 110, 3), (12, 57, 171, 2),
    # a round nearly full, exactly full, and six rounds
    (12, 39, 78, 1), (12, 64, 128, 1), (12, 132, 132, 1),
])
def test_pieces(H, NQ, maxk, want):
    assert _pieces(H, NQ, maxk) == want
