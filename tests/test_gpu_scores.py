"""The product of queries and keys that quantises on the way in, at its edges: rows around the 128-row panel and the 32 rows of a
wavefront, columns around the 64-column step, rows of y that start anywhere in a 128-byte line, contractions that fill the 64- or
128-k loops or leave zeros behind, runs of steps that cut panels and cross products, operands shared between products, blocks of inf,
NaN and zeros; nothing written outside y.  And the calls that take it against the same call by the other route."""
import pytest
import torch

import oracle
from helpers import PRESETS

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
GUARD = 512


def _operand(g, *shape):
    x = torch.randn(*shape, generator=g).to(torch.bfloat16)
    flat = x.view(-1, 32)
    flat[torch.randint(0, flat.shape[0], (flat.shape[0] // 50 + 1,), generator=g)] = 0.0
    return x


def _reference(a, w, tag, quantise_a=True):
    """float64 product of the checker's quantised operands, and its bound: fp32 sums of at most 128 products of exact operands
    (128 * 2^-24 of the sum of magnitudes), then the rounding to bfloat16 (2^-8 of the result; once more on results below 2^-126)."""
    e, m = PRESETS[tag]
    aq = (oracle.qdq_mxfp(a, 32, e, m) if quantise_a else a).double().view(a.shape)
    wq = oracle.qdq_mxfp(w, 32, e, m).double().view(w.shape)
    ref = torch.matmul(aq, wq.transpose(-1, -2))
    return ref, 128 * 2.0 ** -24 * torch.matmul(aq.abs(), wq.abs().transpose(-1, -2)) + 2.0 ** -8 * ref.abs() + 2.0 ** -133


def _run(a, w, tag, quantise_w, M, N, K, Z, a_stride, w_stride, phase=0, quantise_a=True):
    """Through the C entry, y `phase` bytes behind a 128-byte line, sentinels on both sides."""
    from mase_hip import _lib

    e, m = PRESETS[tag] if quantise_a else (0, 0)
    buf = torch.full((GUARD + phase // 2 + Z * M * N + GUARD,), 7.0, dtype=torch.bfloat16, device=DEV)
    first = GUARD + phase // 2
    y = buf[first:first + Z * M * N]
    rc = _lib.load().mase_hip_mxfp_scores(a.data_ptr(), e, m, w.data_ptr(), int(quantise_w), y.data_ptr(), M, N, K, Z, a_stride, w_stride, M * N,
                                          _lib.stream_ptr(a.device))
    assert rc == 0
    assert (buf[:first] == 7.0).all() and (buf[first + Z * M * N:] == 7.0).all(), "written outside y"
    return y.view(Z, M, N).cpu().double()


@pytest.mark.parametrize("phase", [0, 16, 80])
@pytest.mark.parametrize("Z,M,N,K", [
    (1, 1, 8, 32), (1, 1, 64, 128), (2, 31, 72, 64), (3, 32, 56, 96), (2, 33, 128, 128), (1, 127, 136, 64), (2, 128, 192, 32), (1, 129, 200, 128),
    (3, 160, 104, 96), (2, 257, 1000, 128), (1, 300, 520, 64), (40, 200, 520, 128), (9, 1000, 264, 96),
])
def test_scores_against_float64(Z, M, N, K, phase):
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFPMeta

    g = torch.Generator().manual_seed(M * 1000 + N + K)
    tags = list(PRESETS)
    for tag in tags if Z * M * N < 100000 else [tags[(M + phase) % len(tags)]]:
        a, w = _operand(g, Z, M, K), _operand(g, Z, N, K)
        ref, bound = _reference(a, w, tag)
        e, m = PRESETS[tag]
        ad, wd = a.to(DEV), w.to(DEV)
        wq = mxk.quantize_dequantize(wd.reshape(-1), MXFPMeta(32, 8, e, m, True, "rn"), torch.bfloat16)
        got = _run(ad, wq, tag, False, M, N, K, Z, M * K, N * K, phase)
        assert ((got - ref).abs() <= bound).all(), (tag, "W quantised before")
        got = _run(ad, wd, tag, True, M, N, K, Z, M * K, N * K, phase)
        assert ((got - ref).abs() <= bound).all(), (tag, "W quantised on the way in")
        ref, bound = _reference(a, w, tag, quantise_a=False)
        got = _run(ad, wq, tag, False, M, N, K, Z, M * K, N * K, phase, quantise_a=False)
        assert ((got - ref).abs() <= bound).all(), (tag, "A as it is")


@pytest.mark.parametrize("quantise_w", [False, True])
def test_scores_shared_operands(quantise_w):
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn

    g = torch.Generator().manual_seed(5)
    Z, M, N, K = 5, 140, 328, 64
    a, w = _operand(g, Z, M, K), _operand(g, Z, N, K)
    prep = (lambda t: t) if quantise_w else (lambda t: mxk.quantize_dequantize(t.reshape(-1), MXFP8_E4M3_fn, torch.bfloat16))
    ref, bound = _reference(a[:1], w, "MXFP8_E4M3_fn")
    assert ((_run(a.to(DEV), prep(w.to(DEV)), "MXFP8_E4M3_fn", quantise_w, M, N, K, Z, 0, N * K) - ref).abs() <= bound).all()
    ref, bound = _reference(a, w[:1], "MXFP8_E4M3_fn")
    assert ((_run(a.to(DEV), prep(w[:1].to(DEV)), "MXFP8_E4M3_fn", quantise_w, M, N, K, Z, M * K, 0) - ref).abs() <= bound).all()


@pytest.mark.parametrize("quantise_w", [False, True])
@pytest.mark.parametrize("tag", list(PRESETS))
def test_scores_special_blocks(tag, quantise_w):
    """inf and NaN blocks on either side poison exactly the rows and columns that the quantised operands' product has them in."""
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFPMeta

    g = torch.Generator().manual_seed(6)
    Z, M, N, K = 2, 150, 136, 96
    a, w = _operand(g, Z, M, K), _operand(g, Z, N, K)
    a[0, 3, 40], a[1, 149, 95], w[0, 7, 0], w[1, 135, 64] = float("inf"), float("nan"), float("-inf"), float("nan")
    a[0, 5, 32:64], w[1, 9, :32] = 1e-40, 1e30               # (32 products of 1e30 and a few units stay inside fp32: no infinity of the sum's own)
    e, m = PRESETS[tag]
    ref, bound = _reference(a, w, tag)
    wd = w.to(DEV) if quantise_w else mxk.quantize_dequantize(w.to(DEV).reshape(-1), MXFPMeta(32, 8, e, m, True, "rn"), torch.bfloat16)
    got = _run(a.to(DEV), wd, tag, quantise_w, M, N, K, Z, M * K, N * K)
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    ok = ref.isfinite()
    assert ((got - ref).abs() <= bound)[ok].all() and ok.float().mean() > 0.8


@pytest.mark.parametrize("shape_a,shape_w", [((2, 3, 70, 64), (2, 3, 96, 64)), ((70, 64), (3, 96, 64)), ((2, 1, 70, 64), (2, 3, 96, 64)), ((3, 70, 64), (96, 64)),
                                             ((1, 1, 5, 128), (1, 8, 200, 128)), ((2, 3, 700, 128), (2, 3, 72, 128)), ((4, 1, 64), (4, 77, 64)), ((2, 40, 160), (2, 72, 160)),
                                             ((2, 40, 32), (1, 72, 32))])
@pytest.mark.parametrize("func", ["XqWq", "XWq"])
def test_matmul_transposed_view_against_separate(shape_a, shape_w, func):
    """mxfp_matmul(a, w^T) through whichever route takes it against backend="separate", whose operands are the same values."""
    import mase_hip.mxfp.functional as MX
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn, OCP_MXFP6_E2M3

    g = torch.Generator().manual_seed(len(shape_a) + shape_a[-1])
    a, w = _operand(g, *shape_a).to(DEV), _operand(g, *shape_w).to(DEV)
    for xm in (MXFP8_E4M3_fn, OCP_MXFP6_E2M3):
        for other in (w.transpose(-1, -2), w.transpose(-1, -2).contiguous()):
            got = MX.mxfp_matmul(a, other, xm, MXFP8_E4M3_fn, func, "fused")
            aq = MX.quantize_dequantize(a, -1, xm).double() if func == "XqWq" else a.double()
            wq = MX.quantize_dequantize(w, -1, MXFP8_E4M3_fn).double()
            ref = torch.matmul(aq.cpu(), wq.cpu().transpose(-1, -2))
            assert got.shape == ref.shape and got.dtype == torch.bfloat16 and got.is_contiguous()
            bound = 2.0 ** -8 * ref.abs() + shape_a[-1] * 2.0 ** -24 * torch.matmul(aq.cpu().abs(), wq.cpu().abs().transpose(-1, -2))
            assert ((got.cpu().double() - ref).abs() <= bound).all()


def test_scores_refusals():
    import mase_hip.mxfp.kernels as mxk
    from mase_hip import _lib

    a, w = torch.zeros(4, 128, dtype=torch.bfloat16, device=DEV), torch.zeros(64, 128, dtype=torch.bfloat16, device=DEV)
    y = torch.zeros(4, 64, dtype=torch.bfloat16, device=DEV)

    def call(M=4, N=64, K=128, Z=1, e=4, m=3, qw=0, ws=0, ap=None):
        return _lib.load().mase_hip_mxfp_scores(a.data_ptr() if ap is None else ap, e, m, w.data_ptr(), qw, y.data_ptr(), M, N, K, Z, 0, ws, M * N, _lib.stream_ptr(a.device))

    assert call() == 0 and call(M=0) == 0
    assert call(K=160) == -2 and call(N=60) == -2 and call(K=48) == -1 and call(N=0) == -1 and call(M=-1) == -1
    assert call(e=4, m=2) == -1 and call(e=0, m=0, qw=1) == -1 and call(Z=0) == -1 and call(Z=2, ws=64) == -1 and call(ap=a.data_ptr() + 2) == -1
    assert not mxk.scores_shape_supported(12, 64) and not mxk.scores_shape_supported(64, 256)
