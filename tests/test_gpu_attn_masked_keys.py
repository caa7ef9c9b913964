"""Attention over masked keys: a logit of -inf weighs 0 wherever it lies (the
first half block of the list or of a split unit's piece among the places), and
a query left with no other logit gives NaN, as softmax does."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from test_gpu_ops import DEV, dev_bf16, host_f

pytestmark = pytest.mark.gpu

NQ, NK = 2, 16
KW = dict(heads=1, head_dim=128, q_strides=(128, 128), kv_strides=(128, 128))


def _inputs(masked, seed):
    """q, k, v with channel 0 of q at 1 and of the masked keys at -inf."""
    rng = np.random.default_rng(seed)
    q, k, v = (O.bf16(rng.standard_normal((n * 128, 128)).astype(np.float32))
               for n in (NQ, NK, NK))
    q[:, 0] = 1.0
    k[masked, 0] = -np.inf
    return q, k, v


def _call(entry, q, k, v, keep):
    from flashvsr_sm89_ops import _lib
    from flashvsr_sm89_ops.lcsa.hip_lcsa import (block_index, block_sparse_attention_strided,
                                                 dense_attention_strided)
    out = torch.full_like(q, 5.0)
    index = block_index(keep)
    if entry == "dense":
        return dense_attention_strided(q, k, v, None, out=out, **KW)
    if entry == "whole":  # no workspace: no unit is split
        sel, cnt, maxk = index
        _lib.check(_lib.lib().fvsr_bsa_fwd(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), *(128,) * 6, sel.data_ptr(),
            cnt.data_ptr(), maxk, 1, NQ, NK, 128, 128 ** -0.5, None, None, _lib.stream(q)), entry)
        return out
    kw = {"mask": {}, "index": dict(index=index),
          "map": dict(index=index,
                      q_map=torch.arange(NQ * 128, dtype=torch.int32, device=DEV),
                      kv_map=torch.arange(NK * 128, dtype=torch.int32, device=DEV)),
          # a grid of one window row and column: window order is raster order in each 8 x 8
          "window": dict(index=index, window=(2 * NQ, 8, 8, False))}[entry]
    return block_sparse_attention_strided(q, k, v, keep, out=out, **kw, **KW)


# The units of this size run as four pieces of four blocks (a fully kept row):
# halves at the start, in the middle and at the end of a piece and of the row,
# whole pieces, and all but the last key.
_MASKED = {"first half": range(0, 64), "first block": range(0, 128),
           "piece's first half": range(4 * 128, 4 * 128 + 64),
           "piece's first block": range(4 * 128, 5 * 128),
           "inside a piece": range(6 * 128, 6 * 128 + 64),
           "piece's last half": range(12 * 128 - 64, 12 * 128),
           "last half": range(NK * 128 - 64, NK * 128), "a piece": range(4 * 128, 8 * 128),
           "first and third piece": [*range(0, 512), *range(1024, 1536)],
           "all but the last key": range(NK * 128 - 1)}


@pytest.mark.parametrize("entry", ["whole", "index", "mask", "map", "window", "dense"])
@pytest.mark.parametrize("where", list(_MASKED))
def test_masked_keys_weigh_nothing(where, entry):
    from flashvsr_sm89_ops import _lib
    assert _lib.lib().fvsr_bsa_workspace_floats(1, NQ, NK) == 2 * 4 * (128 * 128 + 256)
    masked = np.array(_MASKED[where])
    q, k, v = _inputs(masked, len(masked))
    keep = np.ones((1, NQ, NK), bool)
    rows = np.ones(NQ * 128, bool)
    if entry != "dense":
        keep[0, 1, 5:] = False  # the second query block's pieces are other blocks
        rows[128:] = not set(range(5 * 128)) <= set(masked.tolist())
    got = host_f(_call(entry, *(dev_bf16(O.bf16_bits(t)) for t in (q, k, v)),
                       torch.from_numpy(keep).to(DEV)))
    seen = np.repeat(keep[0], 128, 0).repeat(128, 1)
    with np.errstate(invalid="ignore"):
        s = np.where(seen, q.astype(np.float64) @ k.T.astype(np.float64) * 128 ** -0.5, -np.inf)
        p = np.exp(s - s.max(1, keepdims=True))
        ref = p / p.sum(1, keepdims=True) @ v.astype(np.float64)
    assert np.isfinite(got[rows]).all()
    # P and the output are rounded to bf16: 2^-9 of the weighted |v| each, the
    # bar of the attention tests
    assert np.abs(got - ref)[rows].max() <= 1e-2 * max(1.0, np.abs(ref[rows]).max())
    assert np.isnan(got[~rows]).all()


@pytest.mark.parametrize("entry", ["whole", "index", "mask", "dense"])
def test_query_of_masked_keys_only(entry):
    """Queries that see nothing but -inf logits give NaN, their neighbours in
    the block and in the wave their own results; a row without blocks zeros."""
    q, k, v = _inputs(np.arange(NK * 128), 9)
    q[::2, 0] = 0.0     # 0 * -inf: NaN logits, NaN as well
    q[1::4, 0] = -1.0   # +inf logits: NaN as well
    keep = np.ones((1, NQ, NK), bool)
    keep[0, 1] = entry == "dense"
    got = host_f(_call(entry, *(dev_bf16(O.bf16_bits(t)) for t in (q, k, v)),
                       torch.from_numpy(keep).to(DEV)))
    assert np.isnan(got[:128]).all()
    assert np.isnan(got[128:]).all() if entry == "dense" else (got[128:] == 0).all()
