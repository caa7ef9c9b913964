"""Dense attention with one and with two query blocks per workgroup: bit for
bit the sparse kernel with every block kept, odd block counts included."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (heads, query blocks, key blocks): one block per workgroup (up to 256, and
# where the pairs' last round is less than half full), two (129 of 257 odd
# blocks in one round; a last round more than half full).
@pytest.mark.parametrize("case", [(1, 1, 1), (12, 21, 2), (1, 257, 2), (2, 129, 1), (4, 131, 1),
                                  (3, 261, 1), (1, 256, 3)])
def test_dense_paths(case):
    from flashvsr_sm89_ops import _lib
    from flashvsr_sm89_ops.lcsa.hip_lcsa import block_index, dense_attention_strided
    H, NQ, NK = case
    HD = H * 128
    g = torch.Generator(device=DEV).manual_seed(NQ)
    q, k, v = (torch.randn(n * 128, HD, generator=g, device=DEV).bfloat16() for n in (NQ, NK, NK))
    a = torch.full(((NQ + 1) * 128, HD), 3.0, dtype=torch.bfloat16, device=DEV)
    b = torch.full_like(a, 3.0)
    dense_attention_strided(q, k, v, None, heads=H, head_dim=128, q_strides=(HD, 128),
                            kv_strides=(HD, 128), out=a[:NQ * 128])
    sel, cnt, maxk = block_index(torch.ones(H, NQ, NK, dtype=torch.bool, device=DEV))
    _lib.check(_lib.lib().fvsr_bsa_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), b.data_ptr(), HD, 128, HD, 128, HD, 128,
        sel.data_ptr(), cnt.data_ptr(), maxk, H, NQ, NK, 128, 128 ** -0.5, None, None,
        _lib.stream(q)), "sparse")
    assert torch.equal(a, b)
    assert bool((a[NQ * 128:] == 3.0).all())
    # the first, a middle and the last query block of the last head against float64
    h = HD - 128
    for i in {0, NQ // 2, NQ - 1}:
        qi = q[i * 128:(i + 1) * 128, h:].double()
        p = torch.softmax(qi @ k[:, h:].double().t().contiguous() / 128 ** 0.5, -1)
        ref = p @ v[:, h:].double()
        assert (a[i * 128:(i + 1) * 128, h:].double() - ref).abs().max() <= 1e-2  # the attention bar
