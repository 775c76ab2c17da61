"""Products through the extension module that are not on the block-scaled route: linears on the components and batched products, against the wrappers' way
(the same kernels: equal bits) and, where the wrappers went through torch.matmul, against float64."""
import pytest
import torch

import oracle
from helpers import PRESETS

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _without_extension(monkeypatch, name):
    """The extension with one function switched off."""
    from mase_hip import _lib

    host = _lib.host()

    class Off:
        def __getattr__(self, n):
            return (lambda *a: None) if n == name else getattr(host, n)

    monkeypatch.setattr(_lib, "_host", Off())


@pytest.mark.parametrize("kind", ["mxfp", "minifloat"])
@pytest.mark.parametrize("layer_type,dtype,x_fmt,w_fmt,shape,N,bias", [
    ("XqWqB", "bfloat16", "E5M2", "E4M3", (2, 1024), 996, True), ("XqWqB", "bfloat16", "E4M3", "E5M2", (3, 50, 4096), 4096, True),
    ("XqWqB", "float32", "E4M3", "E3M2", (29, 1408), 768, False), ("XqWqB", "float32", "E2M3", "E2M1", (600, 512), 256, True),
    ("XWqB", "bfloat16", None, "E4M3", (5, 7, 544), 72, True), ("XWqB", "bfloat16", None, "E5M2", (70, 2048), 1000, False),
    ("XqWqBq", "bfloat16", "E5M2", "E5M2", (9, 96), 40, True),
    ("XqWqBq", "bfloat16", "E5M2", "E4M3", (9, 96), 64, True)])      # (the MXFP layer has its quantised bias as well: whole blocks of 32)
def test_layers_on_the_components(monkeypatch, kind, layer_type, dtype, x_fmt, w_fmt, shape, N, bias):
    import mase_hip.minifloat.layers as ML
    import mase_hip.minifloat.meta as mf
    import mase_hip.mxfp.layers as XL
    import mase_hip.mxfp.meta as mx

    g = torch.Generator(device=DEV).manual_seed(N)
    dt, K = getattr(torch, dtype), shape[-1]
    w = (0.5 * torch.randn(N, K, generator=g, device=DEV)).to(dt)
    b = torch.randn(N, generator=g, device=DEV).to(dt) if bias else None
    x = torch.randn(*shape, generator=g, device=DEV).to(dt)
    if kind == "mxfp":
        F = {"E4M3": mx.MXFP8_E4M3_fn, "E5M2": mx.MXFP8_E5M2_fn, "E2M3": mx.OCP_MXFP6_E2M3, "E3M2": mx.OCP_MXFP6_E3M2, "E2M1": mx.OCP_MXFP4_E2M1, None: None}
        bm = mx.OCP_MXFP6_E2M3 if layer_type.endswith("Bq") else None
        if bm is not None:
            b = torch.cat([b, b])[:N // 32 * 32] if N % 32 == 0 else None
        layer = XL.MXFPLinearPTQ(w, b, F[x_fmt], F[w_fmt], bm, layer_type, "fused")
    else:
        F = {"E4M3": mf.FP8_E4M3_fn, "E5M2": mf.FP8_E5M2_fn, "E2M3": mf.FP6_E2M3_fn, "E3M2": mf.FP6_E3M2_fn, "E2M1": mf.FP4_E2M1_fn, None: None}
        layer = ML.MinifloatLinearPTQ(weight=w, bias=b, x_minifloat_meta=F[x_fmt], w_minifloat_meta=F[w_fmt],
                                      b_minifloat_meta=mf.FP8_E4M3_fn if layer_type.endswith("Bq") else None, layer_type=layer_type, backend="fused")
    assert not layer_type.endswith("Bq") or kind == "minifloat" or (layer.b_elements is not None) == (N % 32 == 0)
    first, repeated = layer(x), layer(x)
    assert layer._fast_packed == 3 and first.dtype == dt
    moved = layer(x.transpose(0, 1).contiguous().transpose(0, 1)) if x.dim() > 2 else first       # rows that are not contiguous
    none = layer(x[:0])
    assert none.shape == (0, *shape[1:-1], N) and layer._fast_sig is None
    _without_extension(monkeypatch, "linear_plain")
    want = layer(x)
    assert torch.equal(first, want) and torch.equal(repeated, want) and torch.equal(moved, want)


def test_a_layer_on_the_components_follows_its_weight():
    import mase_hip.mxfp.layers as XL
    import mase_hip.mxfp.meta as mx

    g = torch.Generator(device=DEV).manual_seed(3)
    w, w2 = (torch.randn(96, 256, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    x = torch.randn(4, 256, generator=g, device=DEV).to(torch.bfloat16)
    make = lambda w: XL.MXFPLinearPTQ(w, None, mx.MXFP8_E5M2_fn, mx.MXFP8_E4M3_fn, None, "XqWqB", "fused")      # noqa: E731
    layer, other = make(w), make(w2)
    layer(x)
    layer.load_state_dict(other.state_dict())
    assert torch.equal(layer(x), other(x))
    layer.backend = "separate"
    assert ((layer(x).double() - other(x).double()).norm() / other(x).double().norm()).item() <= 1e-3
    layer.backend, layer.x_mxfp_meta = "fused", mx.OCP_MXFP4_E2M1
    assert not torch.equal(layer(x), other(x))


# keys as a transposed view with rows of outputs of every alignment (K = 64, 96, 128), values as they lie, two formats, dense left operands, fp32
@pytest.mark.parametrize("batch,M,K,N,lying,l_fmt,r_fmt,dtype", [
    ((2, 3), 5, 64, 82, True, "E4M3", "E4M3", "bfloat16"), ((1, 8), 133, 64, 133, True, "E4M3", "E4M3", "bfloat16"), ((2, 4), 2, 128, 1603, True, "E3M2", "E3M2", "bfloat16"),
    ((3,), 1, 128, 65, True, "E5M2", "E5M2", "bfloat16"), ((2, 2), 257, 96, 259, True, "E2M1", "E2M1", "bfloat16"), ((4,), 70, 160, 12, True, "E4M3", "E4M3", "bfloat16"),
    ((1, 8), 96, 96, 128, False, "E3M2", "E3M2", "bfloat16"), ((2, 8), 2, 192, 64, False, "E5M2", "E2M3", "bfloat16"), ((3,), 1000, 2048, 64, False, "E4M3", "E4M3", "bfloat16"),
    ((2,), 33, 64, 7, False, "E4M3", "E4M3", "bfloat16"), ((2, 2), 40, 64, 48, False, None, "E4M3", "bfloat16"), ((2, 2), 40, 128, 50, True, None, "E2M3", "bfloat16"),
    ((2, 2), 24, 64, 36, False, "E4M3", "E4M3", "float32")])
def test_batched_products(monkeypatch, batch, M, K, N, lying, l_fmt, r_fmt, dtype):
    import mase_hip.mxfp.functional as MX
    import mase_hip.mxfp.meta as mx
    from mase_hip import _lib

    names = {"E4M3": "MXFP8_E4M3_fn", "E5M2": "MXFP8_E5M2_fn", "E2M3": "OCP_MXFP6_E2M3", "E3M2": "OCP_MXFP6_E3M2", "E2M1": "OCP_MXFP4_E2M1"}
    g = torch.Generator().manual_seed(M + N)
    dt = getattr(torch, dtype)
    left = torch.randn(*batch, M, K, generator=g).to(dt)
    held = torch.randn(*batch, N, K, generator=g).to(dt)                      # the blocks of the right operand run along its rows
    right = held.transpose(-1, -2) if lying else held.transpose(-1, -2).contiguous()
    lm, rm = None if l_fmt is None else getattr(mx, names[l_fmt]), getattr(mx, names[r_fmt])
    lq = left.float() if lm is None else oracle.qdq_mxfp(left, 32, *PRESETS[names[l_fmt]]).view(left.shape)
    rq = oracle.qdq_mxfp(held, 32, *PRESETS[names[r_fmt]]).view(held.shape)
    want = (lq.double() @ rq.double().transpose(-1, -2).contiguous()).to(dt).double()
    ld = left.to(DEV)
    rd = held.to(DEV).transpose(-1, -2) if lying else right.to(DEV)
    args = (ld, rd, lm, rm, "XWq" if lm is None else "XqWq", "fused")
    taken = _lib.host().matmul_plain(ld, rd, None if lm is None else lm._codes, rm._codes)
    y = MX.mxfp_matmul(*args)
    assert taken is not None and torch.equal(taken, y) and y.shape == (*batch, M, N) and y.dtype == dt
    err = (y.cpu().double() - want).norm() / want.norm()
    assert err <= (1e-3 if dt == torch.bfloat16 else 1e-6)
    if (M * N * y.element_size()) % 16 == 0:                                   # (others went through torch.matmul before)
        _without_extension(monkeypatch, "matmul_plain")
        assert torch.equal(MX.mxfp_matmul(*args), y)


def test_products_that_torch_follows_stay_with_torch():
    """Batches whose outputs do not all start on 16 bytes went through torch.matmul, which is differentiable in a dense left operand, and still do where that
    shows.  (No backward is run here: it multiplies by a transposed view in bfloat16.)"""
    import mase_hip.mxfp.functional as MX
    import mase_hip.mxfp.meta as mx

    g = torch.Generator(device=DEV).manual_seed(1)
    left, right = (torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16) for s in ((2, 5, 64), (2, 64, 7)))
    product = lambda x: MX.mxfp_matmul(x, right, None, mx.MXFP8_E4M3_fn, "XWq", "fused")      # noqa: E731
    plain = product(left)
    leaf = left.clone().requires_grad_()
    y = product(leaf)
    assert y.grad_fn is not None and not plain.requires_grad
    assert ((y.detach().double() - plain.double()).norm() / plain.double().norm()).item() <= 1e-3
    with torch.no_grad():
        assert torch.equal(product(leaf), plain)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(left, torch.ones_like(left))
        assert torch.autograd.forward_ad.unpack_dual(product(dual)).tangent is not None
    with torch.autocast("cuda", torch.float16):
        assert product(left).dtype == torch.float16
    assert torch.equal(product(left), plain)
