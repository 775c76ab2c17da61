"""Ragged products (N or K no multiple of what the tile kernels take) split over K: odd and even counts of outputs (the arrays of sums are
padded to four), a last share that is shorter, one row, bias and every output type, against float64 on the checker's operands, against the
unsplit call, and with a workspace that is short; shapes that other kernels take stay with them; the call without a caller's workspace."""
import pytest
import torch

import oracle
from helpers import PRESETS

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("MNK,tag", [
    ((1, 699, 7488), "MXFP8_E4M3_fn"),
    ((3, 1673, 3040), "OCP_MXFP4_E2M1"),      # 5019 sums
    ((79, 1673, 3040), "MXFP8_E5M2_fn"),      # an odd number of outputs
    ((129, 130, 4128), "OCP_MXFP6_E3M2"),     # 129 steps
    ((120, 500, 800), "OCP_MXFP6_E2M3"),
    ((300, 1000, 4096), "MXFP8_E4M3_fn"),
    ((257, 4080, 4128), "MXFP8_E4M3_fn"),     # 128 x 128 tiles, five shares (of K = 1056 one tile's whole walk is as short)
])
def test_ragged_split(MNK, tag):
    import mase_hip.mxfp.kernels as mxk
    import mase_hip.mxfp.meta as meta
    from mase_hip import _lib

    M, N, K = MNK
    lib = _lib.load()
    need = lib.mase_hip_mxfp_gemm_workspace_bytes(1, M, N, K)
    pitch = (M * N + 3) // 4 * 4
    assert need > 0 and need % (pitch * 4) == 0 and 2 <= need // (pitch * 4) <= 16 and need <= 1 << 25
    g = torch.Generator().manual_seed(M + N + K)
    e, m = PRESETS[tag]
    a = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w_sc, w_el = oracle.extract_mxfp((0.02 * torch.randn(N, K, generator=g)).to(torch.bfloat16), 32, e, m)
    w = oracle.compose_mxfp(w_sc, w_el, 32, e, m, True, torch.float32).double().view(N, K)
    b = torch.randn(N, generator=g)
    ad, sd, ed, bd = (t.to(DEV) for t in (a, w_sc, w_el, b))
    size = a.double().abs() @ w.abs().t()
    for bias in (None, bd):
        ref = a.double() @ w.t() + (0.0 if bias is None else b.double())
        for odt in (torch.float32, torch.bfloat16, torch.float16):
            # fp32 sums of K exact products in any order (their rounding errors add up as their square root: 8 of them), then the output type's rounding
            bound = 8 * K ** 0.5 * 2.0 ** -24 * size + {torch.float32: 2.0 ** -23, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -10}[odt] * ref.abs() + 2.0 ** -24
            for split_k in (True, False):
                y = mxk.mxfp_gemm(ad, None, None, None, sd, ed, getattr(meta, tag), bias, M, N, K, odt, split_k=split_k)
                assert ((y.cpu().double() - ref).abs() <= bound).all(), (odt, split_k)
    # nothing is written behind y, and a workspace that is short is not used
    unsplit = mxk.mxfp_gemm(ad, None, None, None, sd, ed, getattr(meta, tag), None, M, N, K, torch.float32, split_k=False)
    ws = torch.zeros(need, dtype=torch.uint8, device=DEV)
    y = torch.full((M * N + 64,), 7.0, device=DEV)

    def call(fn, *extra):
        y[:M * N] = 0
        assert fn(ad.data_ptr(), 2, None, None, 0, 0, sd.data_ptr(), ed.data_ptr(), e, m, None, 0, y.data_ptr(), 0, M, N, K, 32, *extra, _lib.stream_ptr(y.device)) == 0
        assert (y[M * N:] == 7.0).all()

    call(lib.mase_hip_mxfp_gemm_ws, ws.data_ptr(), need - 1)
    assert torch.equal(y[:M * N].view(M, N), unsplit) and (ws == 0).all()
    call(lib.mase_hip_mxfp_gemm_ws, ws.data_ptr(), need)
    sums = ws.view(torch.float32).view(-1, pitch)[:, :M * N]
    assert (sums != 0).any(1).all() and ((sums.double().sum(0).view(M, N) - unsplit).norm() / unsplit.norm()).item() <= 2e-6      # every share in its array
    assert ((y[:M * N].view(M, N) - unsplit).norm() / unsplit.norm()).item() <= 2e-6
    call(lib.mase_hip_mxfp_gemm_static_ws)                     # (does not split these: no scratch shared between streams)
    assert torch.equal(y[:M * N].view(M, N), unsplit)


def test_shapes_of_other_kernels_are_not_ragged():
    from mase_hip import _lib

    ws = _lib.load().mase_hip_mxfp_gemm_workspace_bytes
    for M, N, K in ((16, 4096, 4096), (64, 8192, 4096), (100, 14304, 4096), (2000, 4096, 4096), (300, 4096, 1088), (1, 777, 224), (4096, 4100, 4096), (16384, 14330, 4096)):
        assert ws(1, M, N, K) == 0, (M, N, K)


def test_products_that_are_left_whole_ask_for_no_room():
    from mase_hip import _lib

    ws = _lib.load().mase_hip_mxfp_gemm_workspace_bytes
    for M, N, K in ((257, 4080, 1056), (700, 1000, 1024), (1500, 1300, 2048), (2000, 2000, 2080), (16, 2001, 256), (3000, 3001, 4096)):
        assert ws(1, M, N, K) == 0, (M, N, K)
