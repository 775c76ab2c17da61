"""Static check of the kernels that count their own outstanding vector-memory operations (inline-asm loads,
stores and DMAs waited for with hand-written s_waitcnt vmcnt(N)): a register spill would add scratch
loads and stores that those counts do not know about, so these kernels must compile without scratch.
Cross-compiles every GEMM translation unit for gfx950 (no GPU needed; the units compile in parallel)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "mase-triton_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


COUNTED = ("gemm_tall_kernel", "gemm_skinny_kernel", "gemm_mid_kernel", "gemm_wide_kernel", "gemm_rows16_kernel", "gemm_scaled_kernel")
UNITS = {"gemm_w_e4m3": 6, "gemm_w_e5m2": 6, "gemm_w_e2m3": 6, "gemm_w_e3m2": 6, "gemm_w_e2m1": 6, "gemm_scaled": 3}  # unit -> least number of such kernels


def _assembly(unit, folder):
    out = os.path.join(folder, unit + ".s")
    cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", "--cuda-device-only", "-S", os.path.join(CSRC, unit + ".hip"), "-o", out]
    subprocess.run(cmd, check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL, timeout=900)
    with open(out) as f:
        return f.read()


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_counted_wait_kernels_use_no_scratch(tmp_path):
    from concurrent.futures import ThreadPoolExecutor

    with ThreadPoolExecutor(max_workers=6) as ex:
        texts = dict(zip(UNITS, ex.map(lambda u: _assembly(u, str(tmp_path)), UNITS)))
    for unit, text in texts.items():
        names = re.findall(r"^(_ZN4mase\w+):\s*; @", text, re.M)
        scratch = re.findall(r"; ScratchSize: (\d+)", text)
        assert len(names) == len(scratch) > 0, unit
        checked = 0
        for name, size in zip(names, scratch):
            if any(tag in name for tag in COUNTED):
                assert int(size) == 0, f"{unit}: {name} spills ({size} bytes of scratch): its s_waitcnt counts would be wrong"
                checked += 1
        assert checked >= UNITS[unit], f"{unit}: {checked} kernels with counted waits found"
        # M0 carries the LDS address of the DMAs between inline-asm statements: nothing else may write it
        m0_writes = [ln for ln in text.splitlines() if re.search(r"\bm0\b", ln) and not ln.strip().startswith(";")]
        assert all(re.match(r"\s*s_mov_b32 m0, s\d+", ln) for ln in m0_writes), (unit, m0_writes[:5])


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
@pytest.mark.parametrize("unit,tag", [("gemm_short_k", "gemm_short_k_kernel"), ("gemm_scaled", "gemm_scaled_mid_kernel")])
def test_counted_wait_kernels_of_one_unit_use_no_scratch(tmp_path, unit, tag):
    """The same check for the kernels that one translation unit holds for all formats."""
    text = _assembly(unit, str(tmp_path))
    sizes = dict(zip(re.findall(r"^(_ZN4mase\w+):\s*; @", text, re.M), re.findall(r"; ScratchSize: (\d+)", text)))
    sizes = {name: size for name, size in sizes.items() if tag in name}
    assert sizes and all(int(size) == 0 for size in sizes.values()), sizes
    m0_writes = [ln for ln in text.splitlines() if re.search(r"\bm0\b", ln) and not ln.strip().startswith(";")]
    assert all(re.match(r"\s*s_mov_b32 m0, s\d+", ln) for ln in m0_writes), m0_writes[:5]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_counted_waits_of_the_scores_kernel_use_no_scratch(tmp_path):
    """Of the attention-scores kernel (template arguments: format, quantise A, quantise W, K) the builds whose W is quantised before fetch it by
    DMA and count their operations; those that quantise W wait with the compiler's own counts (at K = 128 they do use scratch)."""
    text = _assembly("gemm_scores", str(tmp_path))
    sizes = dict(zip(re.findall(r"^(_ZN4mase\w+):\s*; @", text, re.M), re.findall(r"; ScratchSize: (\d+)", text)))
    counted = {name: size for name, size in sizes.items() if re.search(r"mxfp_scores_kernelI.*Lb[01]ELb0ELi(64|128)EE", name)}
    assert len(counted) == 12 and all(int(size) == 0 for size in counted.values()), counted      # five formats and A as it is, two lengths of K
    m0_writes = [ln for ln in text.splitlines() if re.search(r"\bm0\b", ln) and not ln.strip().startswith(";")]
    assert all(re.match(r"\s*s_mov_b32 m0, s\d+", ln) for ln in m0_writes), m0_writes[:5]


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_extract_down_the_rows_leaves_room_for_six_wavefronts(tmp_path):
    """mxfp_strided_tile_kernel waits for memory with up to six wavefronts per SIMD: with code that kept a block's values alive beside its codes it had
    three or four and took up to 17 % longer."""
    text = _assembly("cast_kernels", str(tmp_path))
    occupancy = dict(zip(re.findall(r"^(_ZN4mase\w+):\s*; @", text, re.M), re.findall(r"; Occupancy: (\d+)", text)))
    occupancy = {name: int(n) for name, n in occupancy.items() if "mxfp_strided_tile_kernel" in name}
    assert len(occupancy) == 15 and min(occupancy.values()) >= 6, occupancy


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_composing_e5m2_takes_no_comparison_for_each_code(tmp_path):
    """The one format that the convert instruction does not read.  A test of every code's sign made the kernels depend on how the compiler writes it, two
    instructions or three by what else a translation unit holds."""
    probe = tmp_path / "compose.hip"
    probe.write_text(f"""#include "{CSRC}/mase_device.h"
#include "{CSRC}/mxfp_compose.h"
extern "C" __global__ void compose(const uint4* codes, const uint32_t* scales, uint4* out) {{
    uint4 lo, hi;
    mase::Composer<mase::SFmt<5, 2>>(scales[threadIdx.x]).run16(codes[threadIdx.x], lo, hi);
    out[2 * threadIdx.x] = lo;
    out[2 * threadIdx.x + 1] = hi;
}}
""")
    out = str(tmp_path / "compose.s")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S", str(probe),
                    "-o", out], check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL, timeout=300)
    with open(out) as f:
        text = f.read()
    assert text.count("v_cvt_pk_bf16_f32") == 8 and len(re.findall(r"^\s+v_cmp", text, re.M)) <= 1      # (a scale of 2^-127)
