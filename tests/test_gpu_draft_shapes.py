"""Device draft mask at the edges of its score and threshold kernels: head
dims around a lane's 8-channel chunks and the 128-channel pass, key counts
around the 16-block tiles and the 256 a workgroup takes per trip, query counts
that leave the last workgroup short, and time rows around the threshold
kernel's row batches; bit for bit against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_ops import _draft_check, ops, rnd_bits  # noqa: F401  (ops: fixture)

pytestmark = pytest.mark.gpu


# (heads, head dim, query time rows, blocks per time row, key time rows)
@pytest.mark.parametrize("case", [(1, 8, 1, 1, 1), (2, 24, 1, 5, 3), (1, 40, 3, 3, 3),
                                  (2, 136, 1, 17, 1), (1, 256, 1, 2, 8), (1, 128, 1, 65, 4),
                                  (1, 64, 2, 9, 57), (3, 128, 1, 16, 16), (1, 8, 1, 130, 2)])
def test_draft_shapes(ops, case):  # noqa: F811
    H, D, t, nb, tk = case
    NQ, NK = t * nb, tk * nb
    q = rnd_bits((NQ, 128, H * D), seed=NQ + D, scale=3.0)
    k = rnd_bits((NK, 128, H * D), seed=NK + D + 1, scale=3.0)
    local = np.random.default_rng(NQ).random((nb, nb)) < 0.7
    local[np.arange(nb), np.arange(nb)] = True
    for topk in (0, NK, nb * NK // 3, nb * NK):
        _draft_check(ops, q, k, H, t, local, topk)
