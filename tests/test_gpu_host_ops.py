"""The native host side of quantisation and GEMM: the same results as the
general Python path, which every other call form still reaches."""
import pytest
import torch

DEV = "cuda"
pytestmark = pytest.mark.gpu


@pytest.fixture()
def general(monkeypatch):
    """Calls f with the native calls off."""
    from flashvsr_sm89_ops import _lib

    class Off:
        quantize = gemm = staticmethod(lambda *a: None)

    def run(f):
        with monkeypatch.context() as m:
            m.setattr(_lib, "_host", Off)
            return f()
    return run


def _same(a, b):
    if isinstance(a, tuple):
        assert len(a) == len(b)
        for x, y in zip(a, b):
            _same(x, y)
        return
    assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride()
    assert a.device == b.device and a.requires_grad == b.requires_grad
    v = torch.uint8 if a.element_size() == 1 else torch.int16 if a.element_size() == 2 else torch.int32
    assert torch.equal(a.view(v), b.view(v))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("form", ["plain", "rows", "columns", "empty", "param", "transposed"])
def test_quantize_forms(general, dtype, form):
    from flashvsr_sm89_ops import _lib
    from flashvsr_sm89_ops.fp8_ffn import fused_gelu_quant_fp8
    from flashvsr_sm89_ops.fp8_quant import quantize_fp8
    x = torch.randn(37, 96, device=DEV).to(dtype)
    x = {"plain": x, "rows": x[:, :40], "columns": x[:, 8:48], "empty": x[:0],
         "param": torch.nn.Parameter(x, requires_grad=False), "transposed": x.t()}[form]
    native = _lib.host().quantize(x, True, False) is not None
    assert native == (form not in ("empty", "transposed"))
    for f in (quantize_fp8, fused_gelu_quant_fp8):
        for per_token in (False, True):
            _same(f(x, per_token=per_token), general(lambda: f(x, per_token=per_token)))


def test_gemm_forms(general):
    import flashvsr_sm89_ops as fv
    from flashvsr_sm89_ops import _lib
    M, N, K = 70, 96, 256
    x8, s = fv.quantize_fp8(torch.randn(M, K, device=DEV).bfloat16(), per_token=True)
    w8, ws = fv.quantize_weight_fp8(torch.randn(N, K, device=DEV).bfloat16(), per_channel=True)
    b = torch.randn(N, device=DEV).bfloat16()
    one, one0 = s[:1].reshape(1), ws[0]
    hmax = torch.empty(M, 1, device=DEV)
    wide = torch.zeros(M, 2 * K, device=DEV).to(torch.float8_e4m3fn)
    wide[:, :K] = x8
    forms = [((x8, s, w8, ws, b), {}, True), ((x8, s, w8, ws, None), {}, True),
             ((x8, one, w8, one0, b), {}, True), ((x8[:1], s[:1], w8, ws, b), {}, True),
             ((wide[:, :K], s, w8, ws, b), {}, True), ((x8[:0], s[:0], w8, ws, b), {}, None),
             ((x8, s, w8, ws, b.float()), {}, False), ((x8, s.double(), w8, ws, b), {}, False),
             ((x8, s, w8, ws, b), dict(epilogue=_lib.EPI_ROWMAX, amax_part=hmax), True),
             ((x8, s, torch.nn.Parameter(w8, requires_grad=False), ws, b), {}, True)]
    for args, kw, native in forms:
        if native is not None:
            got = _lib.host().gemm(*args, kw.get("amax_part"))
            assert (got is not None) == native
        a = fv.fp8_gemm(*args, **kw)
        part = hmax.clone()
        _same(a, general(lambda: fv.fp8_gemm(*args, **kw)))
        assert torch.equal(part, hmax)


def test_refusals_and_modes(general):
    """What the general path refuses stays refused with its own error; calls
    under a torch mode go through the general path."""
    import flashvsr_sm89_ops as fv
    from flashvsr_sm89_ops import _lib
    x8, s = fv.quantize_fp8(torch.randn(64, 256, device=DEV).bfloat16(), per_token=True)
    w8, ws = fv.quantize_weight_fp8(torch.randn(96, 256, device=DEV).bfloat16(), per_channel=True)
    bad = [(x8[:, :128], s, w8, ws), (x8, s[:7], w8, ws), (x8, s, w8, ws[:5]),
           (x8.view(torch.uint8), s, w8, ws), (x8, s, w8, ws, s.reshape(-1)[:64]),
           (x8, s.cpu(), w8, ws), (x8[:, 8:], s, w8[:, 8:], ws)]  # the last: unaligned rows
    for args in bad:
        kinds = []
        for call in (lambda: fv.fp8_gemm(*args), lambda: general(lambda: fv.fp8_gemm(*args))):
            with pytest.raises((ValueError, TypeError, RuntimeError)) as e:
                call()
            kinds.append((e.type, str(e.value)))
        assert kinds[0] == kinds[1]
    # a granularity without a truth value: the exception of asking for it
    for call in (lambda f: f(), general):
        with pytest.raises(RuntimeError, match="ambiguous"):
            call(lambda: fv.quantize_fp8(torch.zeros(4, 8, device=DEV), torch.ones(2)))
    with pytest.raises(TypeError):
        fv.quantize_fp8(torch.zeros(4, 8, device=DEV, dtype=torch.int32))
    with pytest.raises(ValueError):
        fv.quantize_fp8(torch.zeros(4, 8, 2, device=DEV, dtype=torch.bfloat16))
    from torch.utils._python_dispatch import TorchDispatchMode

    class Seen(TorchDispatchMode):
        n = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.n += 1
            return func(*args, **(kwargs or {}))

    x = torch.randn(8, 64, device=DEV).bfloat16()
    want = fv.quantize_fp8(x, per_token=True)
    with Seen() as m:
        assert _lib.host().quantize(x, True, False) is None
        got = fv.quantize_fp8(x, per_token=True)
    assert m.n > 0
    _same(got, want)


@pytest.fixture()
def stub():
    """Binds the native calls to a stand-in for the library's quantisation and
    GEMM that launches nothing and returns the status it is given."""
    import ctypes

    from flashvsr_sm89_ops import _lib
    host, L = _lib.host(), _lib.lib()
    names = ("fvsr_quant_workspace_floats", "fvsr_quant_fp8_dt", "fvsr_fp8_gemm",
             "fvsr_gemm_amax_parts")
    real = [ctypes.cast(getattr(L, n), ctypes.c_void_p).value for n in names]
    held = []

    def bind(status):
        calls = []
        for i in (1, 2):
            args, res = _lib._SIGS[names[i]]
            held.append(ctypes.CFUNCTYPE(res, *args)(lambda *a: (calls.append(1), status)[1]))
        addr = [ctypes.cast(f, ctypes.c_void_p).value for f in held[-2:]]
        host.bind(real[0], *addr, real[3])
        return calls
    yield bind
    host.bind(*real)


def test_hip_errors_are_raised(stub):
    """A HIP error is raised by the call that met it, as the general path does,
    and the call is not made again; a refusal goes to the general path."""
    import flashvsr_sm89_ops as fv
    from flashvsr_sm89_ops import _lib
    from flashvsr_sm89_ops.fp8_ffn import fused_gelu_quant_fp8
    x = torch.randn(64, 256, device=DEV).bfloat16()
    x8, s = fv.quantize_fp8(x, per_token=True)
    w8, ws = fv.quantize_weight_fp8(torch.randn(96, 256, device=DEV).bfloat16(), per_channel=True)
    y = fv.fp8_gemm(x8, s, w8, ws)
    calls = [("quantize_fp8", lambda: fv.quantize_fp8(x, per_token=True), (x8, s)),
             ("fused_gelu_quant_fp8", lambda: fused_gelu_quant_fp8(x, per_token=True), None),
             ("fp8_gemm", lambda: fv.fp8_gemm(x8, s, w8, ws), y)]
    for what, f, want in calls:
        n = stub(_lib.FVSR_EHIP)
        with pytest.raises(RuntimeError, match=f"{what} failed: HIP launch error .status -2"):
            f()
        assert len(n) == 1
        for status in (_lib.FVSR_EINVAL, _lib.FVSR_EUNSUPPORTED, _lib.FVSR_EWORKSPACE):
            n = stub(status)
            got = f()
            assert len(n) == 1 and (want is None or _same(got, want) is None)


def test_streams():
    """The launches follow torch's current stream: their inputs are written on a
    side stream behind some milliseconds of other work, other data each time,
    and the work is still running when the calls have returned."""
    import flashvsr_sm89_ops as fv
    side = torch.cuda.Stream()
    big = torch.randn(8192, 8192, device=DEV).bfloat16()
    w8, ws = fv.quantize_weight_fp8(torch.randn(96, 1536, device=DEV).bfloat16(), per_channel=True)
    xs = [torch.randn(2048, 1536, device=DEV).bfloat16() * (i + 1) for i in range(3)]
    want = []
    for x in xs:
        x8, s = fv.quantize_fp8(x)
        want.append((x8, s, fv.fp8_gemm(x8, s, w8, ws)))
    y, z8, zs = torch.zeros_like(xs[0]), torch.zeros_like(want[0][0]), torch.ones_like(want[0][1])
    big @ big
    torch.cuda.synchronize()
    for x, (x8, s, h) in zip(xs, want):
        written = torch.cuda.Event()
        with torch.cuda.stream(side):
            for _ in range(8):
                big @ big
            y.copy_(x)
            z8.copy_(x8)
            zs.copy_(s)
            written.record()
            got = fv.quantize_fp8(y)
            g = fv.fp8_gemm(z8, zs, w8, ws)
        assert not written.query(), "the inputs were there before the calls were made"
        side.synchronize()
        _same(got, (x8, s))
        _same(g, h)
