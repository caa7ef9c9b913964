"""Sparse attention whose units are split over several workgroups (calls that
do not fill the GPU evenly) against the unsplit kernel and the oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from test_gpu_ops import DEV, _attn_check, dev_bf16, host_f

pytestmark = pytest.mark.gpu


def _plan(H, NQ, NK):
    """Floats of partial results of a call (0: nothing split)."""
    from flashvsr_sm89_ops import _lib
    return int(_lib.lib().fvsr_bsa_workspace_floats(H, NQ, NK))


def _unsplit(q, k, v, out, index, H, maps=None, window=None):
    """The same call without a workspace: one workgroup per unit."""
    from flashvsr_sm89_ops import _lib
    sel, cnt, maxk = index
    NQ, NK = cnt.shape[1], maxk
    HD = H * 128
    head = (q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), HD, 128, HD, 128, HD, 128,
            sel.data_ptr(), cnt.data_ptr(), maxk, H, NQ, NK, 128, 128 ** -0.5)
    L = _lib.lib()
    if window is not None:
        rc = L.fvsr_bsa_fwd_window(*head, *window, _lib.stream(q))
    else:
        m = (None, None) if maps is None else tuple(t.data_ptr() for t in maps)
        rc = L.fvsr_bsa_fwd(*head, *m, _lib.stream(q))
    _lib.check(rc, "unsplit attention")
    return out


# (heads, query blocks, key blocks): all units split (fewer than the 256 CUs),
# a split tail behind whole units, pieces of the smallest size, one unit.
@pytest.mark.parametrize("mode", ["direct", "map", "window"])
@pytest.mark.parametrize("case", [(12, 9, 36), (4, 4, 16), (1, 1, 8), (3, 1, 64), (12, 24, 24)])
def test_split_units(case, mode):
    from flashvsr_sm89_ops.lcsa.hip_lcsa import block_index, block_sparse_attention_strided
    H, NQ, NK = case
    assert _plan(H, NQ, NK) > 0
    HD = H * 128
    rng = np.random.default_rng(NQ + NK)
    q, k, v = (O.bf16(rng.standard_normal((n * 128, HD)).astype(np.float32))
               for n in (NQ, NK, NK))
    keep = O.random_block_mask(H, NQ, NK, 0.5, seed=NK)
    if H * NQ > 1:
        keep[0, 0] = False                   # an empty row: zeros
    if NQ > 1:
        keep[H - 1, NQ - 1] = False          # fewer kept blocks than pieces
        keep[H - 1, NQ - 1, NK - 1] = True
        keep[H - 1, 0] = True
    ref = O.sparse_attention(q.reshape(-1, H, 128), k.reshape(-1, H, 128), v.reshape(-1, H, 128),
                             keep)
    perm, kw, raw = np.arange(NQ * 128), {}, {}
    qs, ks, vs = q, k, v
    if mode == "map":
        perm, pk = rng.permutation(NQ * 128), rng.permutation(NK * 128)
        qs, ks, vs = np.empty_like(q), np.empty_like(k), np.empty_like(v)
        qs[perm], ks[pk], vs[pk] = q, k, v
        maps = [torch.from_numpy(m.astype(np.int32)).to(DEV) for m in (perm, pk)]
        kw, raw = dict(q_map=maps[0], kv_map=maps[1]), dict(maps=maps)
    elif mode == "window":
        from flashvsr_sm89_ops.block import window_token_map
        grid = (2, 8, 8 * NQ)
        perm = window_token_map(*grid).numpy()
        qs = np.empty_like(q)
        qs[perm] = q
        kw, raw = dict(window=(*grid, False)), dict(window=(*grid, 0))
    qd, kd, vd = (dev_bf16(O.bf16_bits(t)) for t in (qs, ks, vs))
    index = block_index(torch.from_numpy(keep).to(DEV))
    outs = []
    for _ in range(2):
        out = torch.full((NQ * 128 + 8, HD), 3.0, dtype=torch.bfloat16, device=DEV)
        block_sparse_attention_strided(qd, kd, vd, None, None, heads=H, head_dim=128,
                                       q_strides=(HD, 128), kv_strides=(HD, 128),
                                       out=out[:NQ * 128], index=index, **kw)
        assert bool((out[NQ * 128:] == 3.0).all())
        outs.append(out[:NQ * 128])
    assert torch.equal(outs[0], outs[1])
    got = host_f(outs[0])[perm].reshape(-1, H, 128)
    _attn_check(got, ref)
    assert H * NQ == 1 or (got[:128, 0] == 0).all()
    whole = host_f(_unsplit(qd, kd, vd, torch.empty_like(outs[0]), index, H, **raw))[perm]
    # P and the output are rounded to bf16 in both (2^-9 each), relative to
    # different running maxima
    err = np.linalg.norm(got.reshape(whole.shape) - whole) / np.linalg.norm(whole)
    assert err < 2.0 ** -7
    # ... and the split is no further from the oracle
    r = ref.reshape(whole.shape)
    assert np.linalg.norm(got.reshape(r.shape) - r) <= 1.1 * np.linalg.norm(whole - r)


def test_split_non_finite():
    """A NaN or an infinity in one key block reaches exactly the queries that
    keep it, in a split call as in a whole one."""
    from flashvsr_sm89_ops.lcsa.hip_lcsa import block_index, block_sparse_attention_strided
    H, NQ, NK = 1, 2, 16
    assert _plan(H, NQ, NK) > 0
    g = torch.Generator(device=DEV).manual_seed(3)
    for bad in (float("nan"), float("inf"), -float("inf")):
        q, k, v = (torch.randn(n * 128, 128, generator=g, device=DEV).bfloat16()
                   for n in (NQ, NK, NK))
        k[5 * 128 + 3, 7] = bad
        keep = torch.ones(H, NQ, NK, dtype=torch.bool, device=DEV)
        keep[0, 1, 5] = False
        index = block_index(keep)
        a, b = torch.empty_like(q), torch.empty_like(q)
        block_sparse_attention_strided(q, k, v, None, None, heads=H, head_dim=128,
                                       q_strides=(128, 128), kv_strides=(128, 128), out=a,
                                       index=index)
        _unsplit(q, k, v, b, index, H)
        assert torch.equal(a.isnan(), b.isnan())
        assert torch.isfinite(a[128:]).all()


def test_workspace_checks():
    from flashvsr_sm89_ops import _lib
    L = _lib.lib()
    n = _plan(12, 9, 36)
    t = torch.zeros(36 * 128, 12 * 128, dtype=torch.bfloat16, device=DEV)
    idx = torch.zeros(12 * 9 * 36, dtype=torch.int32, device=DEV)
    ws = torch.empty(n + 4, dtype=torch.float32, device=DEV)
    args = (t.data_ptr(),) * 4 + (1536, 128) * 3 + (idx.data_ptr(), idx.data_ptr(), 36, 12, 9, 36,
                                                     128, 0.1, None, None)
    assert L.fvsr_bsa_fwd_ws(*args, ws.data_ptr(), n - 1, _lib.stream(t)) == _lib.FVSR_EWORKSPACE
    assert L.fvsr_bsa_fwd_ws(*args, ws.data_ptr() + 4, n, _lib.stream(t)) == _lib.FVSR_EUNSUPPORTED
    for units in ((12, 132, 132), (12, 64, 128), (12, 39, 78), (0, 4, 4), (4, 9, 7)):
        assert _plan(*units) == 0


@pytest.mark.parametrize("case", [(1, 1, 1), (2, 3, 63), (2, 5, 64), (1, 4, 257), (3, 2, 600),
                                  (12, 22, 22)])
def test_mask_equals_index(case):
    """A mask given as it is against the same mask through block_index, bit
    for bit: rows of every length around a wave's 64 and a trip's 256 blocks,
    empty and full rows, other types and layouts of the mask."""
    from flashvsr_sm89_ops.lcsa.hip_lcsa import block_index, block_sparse_attention_strided
    H, NQ, NK = case
    HD = H * 128
    g = torch.Generator(device=DEV).manual_seed(NK)
    q, k, v = (torch.randn(n * 128, HD, generator=g, device=DEV).bfloat16() for n in (NQ, NK, NK))
    keep = torch.rand(H, NQ, NK, generator=g, device=DEV) < 0.3
    keep[0, 0] = False
    keep[H - 1, NQ - 1] = True
    wide = torch.zeros(H, NQ, 2 * NK, dtype=torch.bool, device=DEV)
    wide[..., ::2] = keep
    kw = dict(heads=H, head_dim=128, q_strides=(HD, 128), kv_strides=(HD, 128))
    want = torch.empty_like(q)
    block_sparse_attention_strided(q, k, v, None, None, out=want, index=block_index(keep), **kw)
    for m in (keep, keep.to(torch.uint8) * 3, keep.float(), wide[..., ::2]):
        got = torch.full_like(q, 5.0)
        block_sparse_attention_strided(q, k, v, m, None, out=got, **kw)
        assert torch.equal(got, want)


def test_far_rows():
    """K/V rows further apart than 32-bit lane offsets reach (a token stride of
    1.4 GB), through each entry: bit for bit the packed tensors' results."""
    from flashvsr_sm89_ops.lcsa.hip_lcsa import (block_index, block_sparse_attention_strided,
                                                 dense_attention_strided)
    stride = 715827840  # the next multiple of 8 below stays with the lane offsets
    n = 127 * stride + 256
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 2 * n + (8 << 30):
        pytest.skip("needs 190 GB of free GPU memory")
    g = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.randn(m, 128, generator=g, device=DEV).bfloat16() for m in (256, 128, 128))
    far = torch.empty(n, dtype=torch.bfloat16, device=DEV)
    kf, vf = (far.as_strided((128, 128), (stride, 1), c) for c in (0, 128))
    try:
        for t in range(128):
            kf[t] = k[t]
            vf[t] = v[t]
        keep = torch.ones(1, 2, 1, dtype=torch.bool, device=DEV)
        for kw in ({}, {"index": block_index(keep)}, {"index": block_index(keep),
                                                      "window": (2, 8, 16, False)}, None):
            got = []
            for kk, vv, ts in ((k, v, 128), (kf, vf, stride)):
                out = torch.zeros(256, 128, dtype=torch.bfloat16, device=DEV)
                args = dict(heads=1, head_dim=128, q_strides=(128, 128), kv_strides=(ts, 128),
                            out=out)
                if kw is None:
                    dense_attention_strided(q, kk, vv, None, **args)
                else:
                    block_sparse_attention_strided(q, kk, vv, keep, **args, **kw)
                got.append(out)
            assert torch.equal(*got) and bool(got[0].any())
    finally:
        del far, kf, vf
        torch.cuda.empty_cache()
