"""Products of any shape on their own tiles, and products that quantise their dense operand themselves: edges of tiles and steps, every output type, blocks
that take the slow routes."""
import sys
from pathlib import Path

import pytest
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "mase-triton_amd"))
from mase_hip import _lib  # noqa: E402
from mase_hip.mxfp import kernels, meta as mx_meta  # noqa: E402
from mase_hip.mxfp.functional import compose_mxfp_tensor, extract_mxfp_components  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FORMATS = ("MXFP8_E4M3_fn", "MXFP8_E5M2_fn", "OCP_MXFP6_E2M3", "OCP_MXFP6_E3M2", "OCP_MXFP4_E2M1")
# half a unit in the last place, at most 2^-p of the value for p significant bits
HALF_ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}


def _check(y, a, w, bias, out_dtype):
    """fp32 sums of K exact products in any order: errors of 2^-24 of the sums of the magnitudes, adding up as their square root (8 of them), then the
    output type's rounding (and its smallest step)."""
    a, w = a.double(), w.double()
    K = a.shape[-1]
    want = a @ w.transpose(-1, -2).contiguous()
    size = a.abs() @ w.abs().transpose(-1, -2).contiguous()
    if bias is not None:
        want, size = want + bias.double(), size + bias.double().abs()
    fine = want.isfinite()
    assert torch.equal(y.double().isnan()[~fine], want.isnan()[~fine])
    err = (y.double() - want).abs()
    bound = 8 * K ** 0.5 * 2.0 ** -24 * size + 1.01 * HALF_ULP[out_dtype] * want.abs() + 2.0 ** -24
    assert bool((err <= bound)[fine].all()), float((err / bound)[fine].max())


@pytest.mark.parametrize("MNK", [(1, 129, 160), (31, 127, 192), (33, 65, 992), (64, 300, 224), (65, 63, 480), (127, 130, 2016), (129, 257, 416), (200, 1025, 1056),
                                 (700, 641, 288), (1500, 2049, 160)])
@pytest.mark.parametrize("name", FORMATS)
def test_any_shape(MNK, name):
    M, N, K = MNK
    meta = getattr(mx_meta, name)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    w = (0.02 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16)
    bias = torch.randn(N, generator=g, device=DEV)
    sc, el, tm = extract_mxfp_components(w, block_dim=1, mxfp_meta=meta)
    w = compose_mxfp_tensor(sc, el, tm)
    for split_k in (True, False):
        for odt in HALF_ULP:
            for b in (None, bias):
                _check(kernels.mxfp_gemm(a, None, None, None, sc, el, meta, b, M, N, K, odt, split_k=split_k), a, w, b, odt)
    # nothing is written around y, whatever its alignment
    for shift in (0, 1, 2, 8):
        y = torch.full((M * N + 64,), 7.0, dtype=torch.bfloat16, device=DEV)
        _lib.check(_lib.load().mase_hip_mxfp_gemm(a.data_ptr(), 2, None, None, 0, 0, sc.data_ptr(), el.data_ptr(), meta.element_exp_bits, meta.element_frac_bits, None, 0,
                                                  y.data_ptr() + 2 * shift, 2, M, N, K, 32, _lib.stream_ptr(y.device)))
        _check(y[shift:shift + M * N].view(M, N), a, w, None, torch.bfloat16)
        assert bool((y[:shift] == 7.0).all()) and bool((y[shift + M * N:] == 7.0).all())


@pytest.mark.parametrize("odt", [torch.bfloat16, torch.float16])
def test_batch_of_large_odd_products(odt):
    """On the 256 x 256 kernel (test_dispatch_rules.py): the second product's outputs start on an odd multiple of two bytes."""
    B, M, N, K = 2, 4033, 2005, 2368
    meta = mx_meta.MXFP8_E4M3_fn
    g = torch.Generator(device=DEV).manual_seed(9)
    a = torch.randn(B, M, K, generator=g, device=DEV).to(torch.bfloat16)
    sc, el, tm = extract_mxfp_components((0.02 * torch.randn(B * N, K, generator=g, device=DEV)).to(torch.bfloat16), block_dim=1, mxfp_meta=meta)
    w = compose_mxfp_tensor(sc, el, tm).view(B, N, K)
    y = torch.full((B * M * N + 64,), 7.0, dtype=odt, device=DEV)
    _lib.check(_lib.load().mase_hip_mxfp_matmul_batched(a.data_ptr(), sc.data_ptr(), el.data_ptr(), meta.element_exp_bits, meta.element_frac_bits, y.data_ptr() + 32,
                                                        {torch.float16: 1, torch.bfloat16: 2}[odt], M, N, K, B, _lib.stream_ptr(y.device)))
    for b in range(B):
        _check(y[16 + b * M * N:16 + (b + 1) * M * N].view(M, N), a[b], w[b], None, odt)
    assert bool((y[:16] == 7.0).all()) and bool((y[16 + B * M * N:] == 7.0).all())


@pytest.mark.parametrize("shape", [(3, 1, 64, 160), (5, 33, 65, 224), (2, 64, 128, 416), (2, 65, 1, 96), (3, 130, 64, 352), (40, 200, 127, 160), (70, 257, 128, 256)])
@pytest.mark.parametrize("name", FORMATS)
def test_product_that_quantises(shape, name):
    """Against the product of the quantised tensor, with zero blocks, blocks at the ends of the exponent range, inf and NaN in x, and large scales in W."""
    B, M, N, K = shape
    meta = getattr(mx_meta, name)
    e, m = meta.element_exp_bits, meta.element_frac_bits
    g = torch.Generator(device=DEV).manual_seed(sum(shape))
    x = torch.randn(B, M, K, generator=g, device=DEV)
    x *= torch.exp2(torch.randint(-12, 3, (B, M, K), generator=g, device=DEV).float())     # values below the format's range in most blocks
    x[0, 0, :32] = 0.0
    x[0, -1, -32:] *= 2.0 ** -126
    x = x.to(torch.bfloat16)
    w = torch.randn(B * N, K, generator=g, device=DEV).to(torch.bfloat16)
    lib, stream = _lib.load(), _lib.stream_ptr(torch.device(DEV))
    for special in (False, True):
        if special:
            x[1, M // 2, 40] = float("inf")
            x[1, 0, 5] = float("nan")
            w[N - 1, 33] = float("nan")
            w[0, :32] *= 2.0 ** 120
        sc, el, tm = extract_mxfp_components(w, block_dim=1, mxfp_meta=meta)
        xq = kernels.quantize_dequantize(x.view(-1), meta, torch.bfloat16).view(B, M, K)
        y = torch.full((B * M * N + 64,), 7.0, dtype=torch.bfloat16, device=DEV)
        _lib.check(lib.mase_hip_mxfp_matmul_cast(x.data_ptr(), sc.data_ptr(), el.data_ptr(), e, m, y.data_ptr(), M, N, K, B, stream))
        assert bool((y[B * M * N:] == 7.0).all())
        wd = compose_mxfp_tensor(sc, el, tm).view(B, N, K)
        for b in range(B):
            got = y[:B * M * N].view(B, M, N)[b]
            if special and b < 2:                       # (rows or columns of inf and NaN: what the product of the quantised tensor has)
                want = xq[b].double() @ wd[b].double().t().contiguous()
                assert torch.equal(got.isfinite(), want.to(torch.bfloat16).isfinite())
            else:
                _check(got, xq[b], wd[b], None, torch.bfloat16)


def test_refusals():
    lib = _lib.load()
    t = torch.zeros(1 << 16, dtype=torch.uint8, device=DEV)
    p = t.data_ptr()
    assert lib.mase_hip_mxfp_matmul_cast(p, p, p, 4, 3, p, 64, 129, 64, 2, None) == -2
    for call in ((p + 2, 64, 64, 64), (p, 64, 64, 48), (None, 64, 64, 64)):
        assert lib.mase_hip_mxfp_matmul_cast(call[0], p, p, 4, 3, p, *call[1:], 2, None) < 0
    plan = lib.mase_hip_mxfp_matmul_cast_plan
    assert plan(1000, 64, 1024) and plan(5, 64, 96) and not plan(5, 64, 1024) and not plan(1000, 129, 1024) and not plan(1000, 64, 1000)
