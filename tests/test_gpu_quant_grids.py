"""Quantisation at row counts around the grids' edges: the workgroups of the
tensor-mode passes (rows per wave 1 -> 2 -> 3), the table kernels' (one row per
CU and more), a wave's chunk groups, and the partial-maxima reductions."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from test_gpu_ops import DEV, dev_bf16, host_codes, host_f, rnd_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 1536), (255, 64), (256, 520), (257, 1544),
                                       (4095, 16), (4096, 24), (4097, 16), (8193, 40),
                                       (12289, 8), (300, 9224), (1025, 512), (70, 1024),
                                       (70, 1032), (4100, 4600), (4100, 4608)])
def test_tensor_mode_grids(rows, cols, gelu):
    import flashvsr_sm89_ops as ops
    from flashvsr_sm89_ops.fp8_ffn import fused_gelu_quant_fp8
    x = rnd_bits((rows, cols), seed=rows + cols, scale=2.0)
    # the largest magnitude in the last row's last chunk: the edge no pass may miss
    x[-1, -1] = O.bf16_bits(np.float32([37.0]))[0]
    f = fused_gelu_quant_fp8 if gelu else ops.quantize_fp8
    for per_token in (False, True):
        q, s = f(dev_bf16(x), per_token=per_token)
        rq, rs = O.quantize_fp8(x, per_row=per_token, gelu=gelu)
        assert np.array_equal(host_codes(q), rq)
        assert np.array_equal(host_f(s).reshape(-1), rs.reshape(-1))


@pytest.mark.parametrize("rows", [1, 5, 257, 4097])
@pytest.mark.parametrize("low", [False, True])
def test_gelu_tensor_after_rowmax(rows, low):
    """The requantisation after a row-max GEMM: the largest h found from the
    per-slab maxima, or (all h small) by the scan."""
    from flashvsr_sm89_ops import _lib
    cols = 256
    rng = np.random.default_rng(rows)
    h = O.bf16_bits(((-0.75 - 2.0 * rng.random((rows, cols))) if low
                     else rng.standard_normal((rows, cols))).astype(np.float32))
    if not low:
        h[-1, -1] = O.bf16_bits(np.float32([9.0]))[0]
    hd = dev_bf16(h)
    hmax = torch.from_numpy(O.from_bf16_bits(h).reshape(rows, 2, 128).max(2)).contiguous().to(DEV)
    q = torch.empty((rows, cols), dtype=torch.float8_e4m3fn, device=DEV)
    s = torch.zeros(1, dtype=torch.float32, device=DEV)
    n = 2 * int(_lib.lib().fvsr_quant_workspace_floats(rows, cols, 0))
    ws = torch.full((n,), float("nan"), device=DEV)
    _lib.check(_lib.lib().fvsr_gelu_quant_fp8_tensor(hd.data_ptr(), rows, cols, hmax.data_ptr(), 2,
                                                     q.data_ptr(), s.data_ptr(), ws.data_ptr(), n,
                                                     _lib.stream(hd)), "gelu tensor")
    rq, rs = O.quantize_fp8(h, per_row=False, gelu=True)
    assert np.array_equal(host_codes(q), rq) and np.array_equal(host_f(s), rs)
