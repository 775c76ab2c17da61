"""Up to 64 rows on the block-scaled route, on the kernel that each shape names: 64 x 64 tiles (one to 64 rows, columns that fill tiles and
that leave a few, contractions shorter than the ring of eight steps and not multiples of it, K shared by several workgroups with a
shorter last share, more than one round of tiles), and the registers kernel with three operand tiles (33 - 48 rows)."""
import ctypes
import os

import pytest
import torch

import oracle
from helpers import PRESETS

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _plan(M, N, K, may_split, cus=256):
    lib = ctypes.CDLL(os.path.join(ROOT, "mase-triton_amd", "mase_hip", "lib", "libmase_bench.so"))
    lib.mase_bench_scaled_plan.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int] * 2 + [ctypes.c_void_p]
    plan = (ctypes.c_int * 3)()
    assert lib.mase_bench_scaled_plan(M, N, K, cus, may_split, plan) == 0
    return tuple(plan)


@pytest.mark.parametrize("MNK,split_k,plan", [
    ((1, 8, 512), True, (64, 1, 4)),
    ((17, 72, 512), True, (64, 1, 4)),
    ((64, 64, 768), True, (64, 1, 6)),
    ((33, 3000, 1024), True, (64, 1, 8)),
    ((16, 14336, 768), True, (64, 1, 6)),
    ((48, 20000, 1024), True, (64, 1, 8)),         # 313 tiles: a second round
    ((40, 4096, 14336), True, (64, 4, 28)),
    ((50, 1024, 13312), True, (64, 9, 12)),        # 104 steps: 8 x 12 + 8
    ((63, 2176, 10752), True, (64, 7, 12)),
    ((50, 1504, 5120), True, (64, 3, 14)),         # 40 steps: 14, 14, 12
    ((40, 2048, 8192), False, (64, 1, 64)),        # no room for sums
    ((48, 4096, 4096), True, (0, 1, 32)),          # registers kernel, three operand tiles
    ((33, 1000, 3840), True, (0, 1, 30)),
])
def test_few_rows_on_the_kernel_it_names(MNK, split_k, plan):
    import mase_hip.mxfp.kernels as mxk
    import mase_hip.mxfp.meta as meta

    M, N, K = MNK
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    if cus != 256:
        pytest.skip(f"the plans are those of 256 CUs, this device has {cus}")
    assert _plan(M, N, K, split_k) == plan
    g = torch.Generator().manual_seed(M * 3 + N + K)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = (0.02 * torch.randn(N, K, generator=g)).to(torch.bfloat16)
    b = torch.randn(N, generator=g).to(torch.bfloat16)
    x_dq = oracle.qdq_mxfp(x, 32, *PRESETS["OCP_MXFP6_E2M3"]).double().view(M, K)
    w_sc, w_el = oracle.extract_mxfp(w, 32, *PRESETS["OCP_MXFP6_E3M2"])
    w_dq = oracle.compose_mxfp(w_sc, w_el, 32, *PRESETS["OCP_MXFP6_E3M2"], True, torch.float32).double().view(N, K)
    ref = x_dq @ w_dq.t()
    a = mxk.scaled_operand_from_dense(x.to(DEV), meta.OCP_MXFP6_E2M3)
    wop = mxk.scaled_operand_from_mxfp(w_sc.to(DEV), w_el.to(DEV), meta.OCP_MXFP6_E3M2, N, K)
    for bias in (None, b):
        want = ref if bias is None else ref + b.double()
        bd = None if bias is None else b.to(DEV)
        y = mxk.mxfp_gemm_scaled(a, wop, bd, torch.float32, split_k=split_k).cpu().double()
        # the matrix unit adds a block's products with fewer bits than fp32: 1 - 2e-5 of the result in norm (5e-5 held), 1e-3 of the largest anywhere
        assert ((y - want).norm() / want.norm()).item() <= 5e-5
        assert (y - want).abs().max() <= 1e-3 * want.abs().max()
        for odt in (torch.bfloat16, torch.float16):
            y = mxk.mxfp_gemm_scaled(a, wop, bd, odt, split_k=split_k).cpu().double()
            rounded = want.to(odt).double()
            assert ((y - rounded).norm() / rounded.norm()).item() <= 1e-3
