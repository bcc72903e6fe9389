"""Registers of kernels whose number decides how many workgroups share a compute unit or what is spilled, from the compiler's
own figures."""
import os
import re
import subprocess

import pytest

from jvp_flash_attention_amd import build

# kernel, most vector registers (512 per lane and SIMD: 168 for three waves, 256 for two), most bytes spilled
KERNELS = [
    ("bwd2_dkdv_kernel_2wg<__bf16, 64, BWD_PLAIN, MASK_NONE, true, false>", 168, 0),
    ("bwd2_dkdv_kernel_2wg<_Float16, 64, BWD_TANGENT, MASK_NONE, true, false>", 168, 0),
    ("bwd2_dkdv_kernel<__bf16, 64, BWD_PLAIN, MASK_NONE, true, false, false, true>", 168, 0),
    ("bwd2_dkdv_kernel_2wg<__bf16, 64, BWD_DUAL, MASK_NONE, false, true>", 256, 0),
    ("bwd2_dkdv_kernel<__bf16, 64, BWD_DUAL, MASK_BITS, false, true, false>", 256, 0),
    ("fwd3_kernel_2wg<__bf16, 64, true, MASK_NONE, false>", 256, 0),
    ("fwd3_kernel_2wg<_Float16, 64, true, MASK_NONE, false>", 256, 0),
    ("bwd2_both_kernel_2wg<__bf16, 64, BWD_DUAL, MASK_NONE, true>", 256, 0),
    ("bwd2_both_kernel_2wg<__bf16, 64, BWD_DUAL, MASK_BITS, true>", 256, 0),
    ("bwd2_both_kernel_2wg<__bf16, 64, BWD_DUAL, MASK_BITS, false>", 256, 0),
    ("bwd_f32x3_dq_kernel<64, BWD_PLAIN, MASK_NONE, true>", 256, 0),
    ("bwd_f32x3_dq_kernel<64, BWD_PLAIN, MASK_BOOL, true>", 256, 0),
    ("bwd_f32x3_dq_kernel<64, BWD_PLAIN, MASK_ADD, true>", 256, 8),
    ("bwd_f32x3_dq_kernel<64, BWD_TANGENT, MASK_BOOL, true>", 256, 0),
    ("bwdw_dkdv_kernel<__bf16, 256, BWD_PLAIN, MASK_NONE, false, true>", 512, 0),
    ("bwdw_dkdv_kernel<_Float16, 256, BWD_PLAIN, MASK_BOOL>", 512, 80),
    ("bwdw_dkdv_kernel<__bf16, 256, BWD_TANGENT, MASK_ADD, true>", 512, 96),
]


@pytest.fixture(scope="module")
def figures(tmp_path_factory):
    """{kernel: (vector registers, scratch bytes)}, compiled on their own (some ten seconds)."""
    src = tmp_path_factory.mktemp("registers") / "kernels.hip"
    kinds = "".join(f'#include "{h}.hpp"\n' for h in ("fwd_kernel_v3", "bwd_kernel", "bwd_kernel_f32x3", "bwd_kernel_v2", "bwd_kernel_wide"))
    takes = lambda k: "const FwdParams" if k.startswith("fwd") else "const BwdParams, const int" if "_both_" in k else "const BwdParams"  # noqa: E731
    src.write_text(kinds + "namespace jvpfa {\n" + "".join(f"template __global__ void {k}({takes(k)});\n" for k, _, _ in KERNELS) + "}\n")
    asm = str(src) + ".s"
    subprocess.run([build.HIPCC, *build.FLAGS, "-Wno-pass-failed", "-I", build.CSRC, "--cuda-device-only", "-S", str(src), "-o", asm],
                   check=True, capture_output=True)
    with open(asm) as f:
        blocks = re.split(r"\n  - \.agpr_count:", f.read())[1:]
    found = [tuple(int(re.search(rf"\.{k}:\s+(\d+)", b).group(1)) for k in ("vgpr_count", "private_segment_fixed_size")) for b in blocks]
    assert len(found) == len(KERNELS)  # in the order of the text
    return dict(zip((k for k, _, _ in KERNELS), found))


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no HIP compiler")
@pytest.mark.parametrize("kernel,registers,spilled", KERNELS)
def test_registers(figures, kernel, registers, spilled):
    assert figures[kernel][0] <= registers and figures[kernel][1] <= spilled
