"""FP8 GEMM tile shapes against the oracle: the small tiles (64 x 64 to 128 x
256), the 192-row tiles, every K-step remainder of their pipelines and ragged
edges, on an output view whose surroundings must keep a sentinel."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from test_gpu_ops import (DEV, _close_bf16, _gemm_inputs, codes_dev, dev_bf16, host_bits,
                                host_f)

pytestmark = pytest.mark.gpu

# K steps of 128 around the pipelines' depths (trips of 4 or 6 steps).  Which
# kernel a shape reaches depends on the epilogue (row maxima take 64 x 128 where
# the others take 64 x 64); tests/test_gemm_plan.py checks that every kernel is
# reached with each epilogue it has, at every remainder of its trips.
_SHAPES = [(65, 72, 128 * n) for n in (1, 2, 3, 4, 5, 6, 7, 8, 9, 13)]
_SHAPES += [(8200, 72, 128 * n) for n in (1, 2, 3, 4, 5, 6, 7)]       # 64 x 128
_SHAPES += [(8200, 200, 128 * n) for n in (7, 8, 9, 14, 17, 18, 19, 20)]  # 128 x 128
_SHAPES += [(10001, 520, 128 * n) for n in (5, 6, 7, 8, 9, 16, 17)]   # 128 x 256
_SHAPES += [(4001, 1032, 128 * n) for n in (33, 34, 35, 36, 37, 38)]  # ... long K
_SHAPES += [
    (1, 64, 256), (64, 64, 128), (63, 1000, 384), (512, 1536, 1536),   # 64 x 64
    (129, 1544, 640), (1152, 1536, 1536), (1025, 1400, 896),           # 64 x 128
    (2079, 1536, 1536), (1500, 1536, 1664), (2500, 1536, 4224),        # 128 x 128
    (3001, 1280, 4096), (2800, 1536, 4224), (4001, 1536, 4096),        # 128 x 256, long K
    (4001, 2056, 512), (7001, 2056, 768), (8200, 1536, 1792),          # general ring
    (5001, 2056, 4096), (4200, 4600, 1024),
    (3301, 1280, 512), (3301, 1280, 4352),                             # 128-row ring
    (3301, 2560, 512), (6200, 1536, 768), (7000, 1536, 4096), (12300, 1536, 512),  # 192-row
    (8201, 1536, 768), (8449, 4608, 512), (8201, 1536, 4352),          # 256-row, prefetching
]


@pytest.mark.parametrize("epi", ["bias", "rowmax", "gate_add"])
@pytest.mark.parametrize("MNK", _SHAPES)
def test_fp8_gemm_tiles(MNK, epi):
    import flashvsr_sm89_ops as ops
    from flashvsr_sm89_ops import _lib
    M, N, K = MNK
    a, b, sa, sb, bias = _gemm_inputs(M, N, K, seed=M + 7 * N + K)
    args = (codes_dev(a), torch.from_numpy(sa).to(DEV), codes_dev(b), torch.from_numpy(sb).to(DEV),
            dev_bf16(bias))
    ref = O.fp8_gemm(a, sa, b, sb, O.from_bf16_bits(bias),
                     acc_dtype=np.float64 if M * N * K < 1e9 else np.float32)
    buf = torch.full((M + 70, N + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    out, kw = buf[:M, :N], {}
    if epi == "rowmax":
        hmax = torch.full((M + 1, (N + 127) // 128), 9.0, dtype=torch.float32, device=DEV)
        kw = dict(epilogue=_lib.EPI_ROWMAX, amax_part=hmax[:M])
    elif epi == "gate_add":
        gate = torch.linspace(-2, 2, N, device=DEV).to(torch.bfloat16)
        out.copy_(torch.linspace(-4, 4, M * N, device=DEV).reshape(M, N))
        res = out.clone().float()
        kw = dict(epilogue=_lib.EPI_GATE_ADD, res=out, gate=gate)  # in place: c is res
    y = ops.fp8_gemm(*args, out=out, **kw)
    assert bool((buf[M:] == 7.0).all()) and bool((buf[:M, N:] == 7.0).all()), "stray store"
    if epi == "gate_add":
        # bf16(res + bf16(gate * h)) of the bias epilogue's h, bit for bit
        h = ops.fp8_gemm(*args).float()
        want = (res + (gate.float() * h).to(torch.bfloat16).float()).to(torch.bfloat16)
        assert torch.equal(y, want)
        return
    # the bar of the GEMM tests: at most one bf16 ulp, on few elements
    _close_bf16(host_f(y), ref)
    if epi == "rowmax":
        hf = O.from_bf16_bits(host_bits(y.contiguous()))
        for p in range((N + 127) // 128):
            assert np.array_equal(host_f(hmax)[:M, p], hf[:, p * 128:(p + 1) * 128].max(1))
        assert bool((hmax[M] == 9.0).all())


@pytest.mark.parametrize("K", [1536, 4096])
def test_fp8_gemm_rows_do_not_depend_on_the_tile(K):
    """Every tile shape sums K in the same order: the rows of a small product
    are bit for bit the rows of a large one."""
    import flashvsr_sm89_ops as ops
    a, b, sa, sb, bias = _gemm_inputs(8448, 1536, K, seed=K)
    ad, bd = codes_dev(a), codes_dev(b)
    sad, sbd, bi = torch.from_numpy(sa).to(DEV), torch.from_numpy(sb).to(DEV), dev_bf16(bias)
    full = ops.fp8_gemm(ad, sad, bd, sbd, bi)
    for M in (64, 700, 1152, 2079, 4000, 6200):
        assert torch.equal(ops.fp8_gemm(ad[:M], sad[:M], bd, sbd, bi), full[:M])


@pytest.mark.parametrize("M", [300, 2079, 8200])
def test_rowmax_passes_nans_over(M):
    """Row maxima of the row-max epilogue ignore NaN outputs (a NaN bias
    column, a row whose every value is NaN: -inf) and keep infinities."""
    import flashvsr_sm89_ops as ops
    from flashvsr_sm89_ops import _lib
    N, K = 1536, 512
    a, b, sa, sb, bias = _gemm_inputs(M, N, K, seed=M)
    sa[3] = np.nan
    bias = O.from_bf16_bits(bias)
    bias[5], bias[200], bias[1535] = np.nan, np.inf, -np.inf
    hmax = torch.empty((M, N // 128), dtype=torch.float32, device=DEV)
    y = ops.fp8_gemm(codes_dev(a), torch.from_numpy(sa).to(DEV), codes_dev(b),
                     torch.from_numpy(sb).to(DEV), dev_bf16(O.bf16_bits(bias)),
                     epilogue=_lib.EPI_ROWMAX, amax_part=hmax)
    h = host_f(y).reshape(M, N // 128, 128)
    want = np.where(np.isnan(h), -np.inf, h).max(2)
    assert np.array_equal(host_f(hmax), want)
    assert (host_f(hmax)[3] == -np.inf).all() and (np.delete(host_f(hmax), 3, 0)[:, 1] == np.inf).all()
