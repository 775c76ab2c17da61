"""Calls through the extension module against the same calls through the Python wrappers (the module replaced by one that takes no
call): the same values, types, shapes and layouts, or the same error, over contiguous and strided, aligned and misaligned, empty and
0-d inputs, every block axis, dtype, format, round mode and output type; and the calls that the module must leave to the wrappers."""
import sys
import threading
import time
from fractions import Fraction

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


class _TakesNothing:
    def __getattr__(self, name):
        return lambda *args: None


def _both(monkeypatch, fn):
    from mase_hip import _lib

    def run():
        try:
            return fn()
        except Exception as e:                               # the error is the result
            return type(e)

    plain = run()
    with monkeypatch.context() as m:
        m.setattr(_lib, "_host", _TakesNothing())
        general = run()
    return plain, general


def _same(a, b):
    if isinstance(a, torch.Tensor):
        assert isinstance(b, torch.Tensor) and a.dtype == b.dtype and a.shape == b.shape and a.device == b.device and not a.requires_grad and type(a) is type(b)
        assert a.is_contiguous() == b.is_contiguous()
        bits = {1: torch.uint8, 2: torch.int16, 4: torch.int32}[a.element_size()]
        assert torch.equal(a.contiguous().view(bits), b.contiguous().view(bits))
    elif isinstance(a, (tuple, list)):
        assert len(a) == len(b)
        for x, y in zip(a, b):
            _same(x, y)
    else:
        assert a == b, (a, b)


def _inputs():
    g = torch.Generator().manual_seed(1)
    base = torch.randn(64, 96, generator=g).to(DEV)
    big = torch.randn(4 * 64 * 96 + 3, generator=g).to(DEV)
    yield "matrix", base
    yield "3-D", big[:4 * 64 * 96].view(4, 64, 96)
    yield "vector", base.view(-1)[:320]
    yield "transposed", base.t()
    yield "every other row", base[::2]
    yield "offset by one", big[1:1 + 64 * 96].view(64, 96)
    yield "columns that are no whole blocks", big[:32 * 33].view(32, 33)
    yield "no whole blocks at all", big[:33]
    yield "empty", base[:0]
    yield "0-d", base[0, 0]
    yield "one block", base.view(-1)[:32]
    yield "needs a gradient", base.clone().requires_grad_()
    yield "expanded", base[:1].expand(32, 96)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32, torch.float64, torch.int32])
def test_casts_either_way(monkeypatch, dtype):
    import mase_hip.minifloat.functional as MF
    import mase_hip.minifloat.meta as mf
    import mase_hip.mxfp.functional as MX
    import mase_hip.mxfp.meta as mx

    metas = [mx.MXFP8_E4M3_fn, mx.OCP_MXFP4_E2M1, mx.MXFPMeta(16, 8, 3, 2, False, "rz"), mx.MXFPMeta(32, 8, 5, 2, True, "up")]
    fmetas = [mf.FP8_E5M2_fn, mf.MinifloatMeta(3, 4, False, "ru"), mf.MinifloatMeta(2, 1, True, "nearest")]
    for name, x in _inputs():
        x = x.detach().to(dtype) if not x.requires_grad else x.detach().to(dtype).requires_grad_(dtype.is_floating_point)
        if name in ("transposed", "every other row", "offset by one", "expanded") and dtype != torch.float32:
            continue                                          # (.to made them dense)
        for meta in metas:
            for dim in (-1, 0, 1, -2, 5):
                for out in (None, torch.float16, torch.float64):
                    _same(*_both(monkeypatch, lambda: MX.quantize_dequantize(x, dim, meta, out)))
                a, b = _both(monkeypatch, lambda: MX.extract_mxfp_components(x, dim, meta))
                _same(a, b)
                if isinstance(a, tuple):
                    for out in (None, torch.float32, torch.float64):
                        _same(*_both(monkeypatch, lambda: MX.compose_mxfp_tensor(a[0], a[1], a[2], out)))
                    _same(*_both(monkeypatch, lambda: MX.compose_mxfp_tensor(a[0][:-1], a[1], a[2])))
                    _same(*_both(monkeypatch, lambda: MX.compose_mxfp_tensor(a[0], a[1].cpu(), a[2])))
        for meta in fmetas:
            for out in (None, torch.bfloat16, torch.float64):
                _same(*_both(monkeypatch, lambda: MF.quantize_dequantize(x, meta, out)))
            a, b = _both(monkeypatch, lambda: MF.extract_minifloat_component(x, meta))
            if isinstance(a, tuple):
                _same((a[0].view(torch.int16), a[1]), (b[0].view(torch.int16), b[1]))
                _same(*_both(monkeypatch, lambda: MF.compose_minifloat_component(a[0], a[1], None if dtype.is_floating_point else torch.float32)))
                _same(*_both(monkeypatch, lambda: MF.compose_minifloat_component(a[0].view(torch.int16), a[1], torch.float32)))
            else:
                _same(a, b)


@pytest.mark.parametrize("dim", [0.0, 1.0, -1.0, 0.5, torch.tensor(1.0), Fraction(1), True, torch.tensor(1)])
def test_axes_that_are_no_whole_numbers(monkeypatch, dim):
    """An axis that is no integer is refused, whatever it compares equal to; True and a 0-d integer tensor are integers."""
    import mase_hip.mxfp.functional as MX
    from mase_hip import _lib
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as m

    x = torch.randn(64, 64, device=DEV)
    sc, el, tm = MX.extract_mxfp_components(x, -1, m)
    tm = tm.create(block_dim=dim)
    for fn in (lambda: MX.extract_mxfp_components(x, dim, m), lambda: MX.quantize_dequantize(x, dim, m), lambda: MX.compose_mxfp_tensor(sc, el, tm)):
        plain, general = _both(monkeypatch, fn)
        _same(plain, general)
        whole = not isinstance(dim, (float, Fraction)) and not (isinstance(dim, torch.Tensor) and dim.is_floating_point())
        assert whole != (plain is TypeError)
    if not whole:
        assert _lib.host().extract_mxfp(x, dim, m._codes) is None and _lib.host().qdq_mxfp(x, dim, m._codes, None) is None


def test_layers_either_way(monkeypatch):
    import mase_hip.minifloat.layers as ML
    import mase_hip.minifloat.meta as mf
    import mase_hip.mxfp.layers as XL
    import mase_hip.mxfp.meta as mx

    g = torch.Generator().manual_seed(2)
    for bias in (None, torch.randn(520, generator=g).to(DEV), torch.randn(520, generator=g).to(torch.bfloat16).to(DEV)):
        w = torch.randn(520, 512, generator=g).to(torch.bfloat16).to(DEV)     # (of a size that the scale-free formats hold)
        layers = [XL.MXFPLinearPTQ(w, bias, mx.MXFP8_E4M3_fn, mx.OCP_MXFP6_E3M2, None, "XqWqB", "fused"),
                  ML.MinifloatLinearPTQ(weight=w, bias=bias, x_minifloat_meta=mf.FP8_E4M3_fn, w_minifloat_meta=mf.FP6_E2M3_fn, b_minifloat_meta=None,
                                        layer_type="XqWqB", backend="fused")]
        big = torch.randn(300 * 512 + 1, generator=g).to(torch.bfloat16).to(DEV)
        for layer in layers:
            for x in (big[:512].view(1, 512), big[:512], big[:7 * 512].view(7, 1, 512), big[:300 * 512].view(300, 512), big[1:1 + 40 * 512].view(40, 512),
                      big[:64 * 512].view(64, 512)[::2], big[:0].view(0, 512), big[:512].view(1, 512).float(), big[:256].view(1, 256),
                      big[:512].view(1, 512).clone().requires_grad_()):
                try:
                    layer(x)                                  # the first call of a kind goes the general way
                except Exception:
                    pass
                a, b = _both(monkeypatch, lambda: layer(x))
                _same(a, b)
            # written weights are noticed
            x = big[:512].view(1, 512)
            before = layer(x).clone()
            for name in ("w_elements", "w_element"):
                p = getattr(layer, name, None)
                if p is not None:
                    with torch.no_grad():
                        p.copy_(torch.zeros_like(p.view(torch.uint8) if p.dtype == torch.uint8 else p.view(torch.int16)).view(p.dtype))
            assert not torch.equal(layer(x), before)


def test_scores_either_way(monkeypatch):
    import mase_hip.mxfp.functional as MX
    import mase_hip.mxfp.meta as mx

    g = torch.Generator().manual_seed(3)
    q, k = (torch.randn(2, 3, 200, 64, generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
    m = mx.MXFP8_E4M3_fn
    for a, b in ((q, k.transpose(-1, -2)), (q[0, 0], k[0, 0].t()), (q[:, :, :1], k.transpose(-1, -2)), (q, k[:1].transpose(-1, -2)), (q[:, ::2], k[:, ::2].transpose(-1, -2)),
                 (q, k.transpose(-1, -2).contiguous()), (q.float(), k.float().transpose(-1, -2)), (q, k[..., :32].transpose(-1, -2)), (q[0], k.transpose(-1, -2)),
                 (q.transpose(1, 2), k.transpose(-1, -2)), (q[:, :, :0], k.transpose(-1, -2)), (q, k[:, :, :196].transpose(-1, -2))):
        plain, general = _both(monkeypatch, lambda: MX.mxfp_matmul(a, b, m, m, "XqWq", "fused"))
        if isinstance(plain, torch.Tensor):                   # (another kernel sums in another order: a last bit of bfloat16, of sums of 64 products)
            assert plain.shape == general.shape and plain.dtype == general.dtype and plain.is_contiguous()
            d, scale = (plain.double() - general.double()).abs(), general.double().abs()
            assert (d <= 2.0 ** -7 * scale + 1e-4).all()
        else:
            assert plain is general


@pytest.mark.parametrize("shape,N,K,way", [((2, 3, 200), 200, 64, 2), ((300,), 72, 32, 2), ((1, 1, 5), 1000, 128, 2), ((20, 513), 2504, 64, 2), ((9, 640), 1000, 128, 1),
                                           ((2, 24, 300), 512, 96, 0), ((1, 700), 16384, 128, 0), ((2000,), 8192, 96, 0), ((2500, 1), 2000, 96, 2), ((66000, 16), 200, 96, 0)])
def test_scores_each_way(monkeypatch, shape, N, K, way):
    """Each of the three ways through the module and through the wrappers: the same kernels, so the same bits."""
    import mase_hip.mxfp.functional as MX
    import mase_hip.mxfp.kernels as mxk
    from mase_hip import _lib
    from mase_hip.mxfp.meta import OCP_MXFP6_E2M3 as m

    batches = 1
    for d in shape[:-1]:
        batches *= d
    assert mxk.scores_plan(shape[-1], N, K, batches, True) == way
    g = torch.Generator(device=DEV).manual_seed(N + K)
    q, k = (torch.randn(*s, K, generator=g, device=DEV, dtype=torch.bfloat16) for s in (shape, (*shape[:-1], N)))
    k = k.transpose(-1, -2)
    assert (_lib.host().scores(q, k, m._codes) is None) == (batches > 65535 and way == 0)      # (more products than a launch of the general kernels takes)
    _same(*_both(monkeypatch, lambda: MX.mxfp_matmul(q, k, m, m, "XqWq", "fused")))


def test_left_to_the_wrappers():
    """Function and dispatch modes, vmap and other devices see what they saw: the module takes none of these calls."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    import mase_hip.mxfp.functional as MX
    from mase_hip import _lib
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as m

    host, x = _lib.host(), torch.randn(4, 64, device=DEV)
    assert host.qdq_mxfp(x, -1, m._codes, None) is not None
    seen = []

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    for mode in (Functions, Dispatch):
        seen.clear()
        with mode():
            assert host.qdq_mxfp(x, -1, m._codes, None) is None
            y = MX.quantize_dequantize(x, -1, m)
        assert seen and torch.equal(y, MX.quantize_dequantize(x, -1, m))

    class Sub(torch.Tensor):
        pass

    assert host.qdq_mxfp(x.as_subclass(Sub), -1, m._codes, None) is None
    assert host.qdq_mxfp(x.cpu(), -1, m._codes, None) is None and host.qdq_mxfp(None, -1, m._codes, None) is None
    assert host.qdq_mxfp(x.to_sparse(), -1, m._codes, None) is None
    with pytest.raises(RuntimeError):
        MX.quantize_dequantize(x.cpu(), -1, m)
    with pytest.raises(Exception):
        torch.vmap(lambda t: MX.quantize_dequantize(t, -1, m))(x)


def _plain_calls():
    """Each function of the module once, its arguments plain; outputs of at least 32 MB."""
    import mase_hip.minifloat.functional as MF
    import mase_hip.minifloat.meta as mf
    import mase_hip.mxfp.functional as MX
    import mase_hip.mxfp.kernels as mxk
    from mase_hip import _lib
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as m

    host, f8 = _lib.host(), mf.FP8_E4M3_fn
    x = torch.randn(4096, 8192, device=DEV)
    sc, el, _ = MX.extract_mxfp_components(x, -1, m)
    codes, _ = MF.extract_minifloat_component(x, f8)
    a = torch.randn(4096, 512, device=DEV).to(torch.bfloat16)
    w = mxk.scaled_operand_from_mxfp(*MX.extract_mxfp_components(a, -1, m)[:2], m, 4096, 512)
    q, k = (torch.randn(32, 1024, 64, device=DEV).to(torch.bfloat16) for _ in range(2))
    return {"extract_mxfp": lambda: host.extract_mxfp(x, -1, m._codes), "extract_mxfp, rows": lambda: host.extract_mxfp(x, 0, m._codes),
            "qdq_mxfp": lambda: host.qdq_mxfp(x, -1, m._codes, None), "compose_mxfp": lambda: host.compose_mxfp(sc, el, m._codes, 0, (4096, 8192)),
            "minifloat, extract": lambda: host.minifloat(0, x, f8._codes, None), "minifloat, compose": lambda: host.minifloat(1, codes, f8._codes, 0),
            "minifloat, both": lambda: host.minifloat(2, x, f8._codes, None),
            "linear_scaled": lambda: host.linear_scaled(a, 4, 3, 0, w.codes, w.scales, 4096, None),
            "scores": lambda: host.scores(q, k.transpose(-1, -2), m._codes)}


def test_other_threads_run_beside_a_call():
    """A call lets go of the interpreter while it allocates and launches: with the interpreter's own switching put off, another thread gets
    on only where a call lets it.  Every output is kept, so every call waits for the driver to allocate."""
    calls = _plain_calls()
    ticks, stop = [0], threading.Event()

    def tick():
        while not stop.is_set():
            ticks[0] += 1
            time.sleep(1e-4)

    interval = sys.getswitchinterval()
    thread = threading.Thread(target=tick)
    thread.start()
    try:
        sys.setswitchinterval(1000.0)
        for name, call in calls.items():
            torch.cuda.empty_cache()
            before, kept = ticks[0], [call() for _ in range(16)]
            seen = ticks[0] - before
            assert seen > 0, name
            assert all(y is not None for y in kept), name
            del kept
    finally:
        sys.setswitchinterval(interval)
        stop.set()
        thread.join()


@pytest.mark.parametrize("take", range(9))
def test_the_module_takes_plain_calls(take):
    """(Where it took none, both sides of the comparisons above would be the wrappers.)"""
    name, call = list(_plain_calls().items())[take]
    assert call() is not None, name


@pytest.mark.parametrize("kind", ["mxfp", "minifloat"])
def test_layers_go_through_the_module(monkeypatch, kind):
    """From the second call of a kind on; again after a call of another look."""
    import mase_hip.minifloat.layers as ML
    import mase_hip.minifloat.meta as mf
    import mase_hip.mxfp.layers as XL
    import mase_hip.mxfp.meta as mx
    from mase_hip import _lib

    w = torch.randn(520, 512, device=DEV).to(torch.bfloat16)
    layer = (XL.MXFPLinearPTQ(w, None, mx.MXFP8_E4M3_fn, mx.OCP_MXFP6_E3M2, None, "XqWqB", "fused") if kind == "mxfp" else
             ML.MinifloatLinearPTQ(weight=w, bias=None, x_minifloat_meta=mf.FP8_E4M3_fn, w_minifloat_meta=mf.FP6_E2M3_fn, b_minifloat_meta=None, layer_type="XqWqB",
                                   backend="fused"))
    host, seen = _lib.host(), []

    class Watched:
        def __getattr__(self, name):
            def call(*args):
                y = getattr(host, name)(*args)
                if name == "linear_scaled":
                    seen.append(y)
                return y
            return call

    monkeypatch.setattr(_lib, "_host", Watched())
    for rows, calls in ((3, 0), (3, 1), (3, 2), (70, 2), (70, 3), (3, 3), (3, 4)):
        y = layer(torch.randn(rows, 512, device=DEV).to(torch.bfloat16))
        assert len(seen) == calls
        assert seen == [] or all(t is not None for t in seen)
        if calls and rows == 3 and calls in (1, 2, 4):
            assert y is seen[-1]


def test_streams_and_capture():
    """The call runs on the current stream, also while it is captured."""
    import mase_hip.mxfp.functional as MX
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as m

    x = torch.randn(256, 512, device=DEV).to(torch.bfloat16)
    want = MX.quantize_dequantize(x, -1, m)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        sc, el, tm = MX.extract_mxfp_components(x, -1, m)
        y = MX.compose_mxfp_tensor(sc, el, tm)
    for seed in range(3):
        x.copy_(torch.randn(256, 512, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), MX.quantize_dequantize(x, -1, m).view(torch.int16))
    assert want.shape == y.shape
