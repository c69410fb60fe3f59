"""The machine code of the library's own kernels, read from the build: wait states the compiler cannot see are needed,
because the lane swaps sit in assembly statements."""
import os
import re
import subprocess

import pytest

BUILD = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mcmc-bnn-example_amd", "build")
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
# wait states between a matrix instruction of up to eight passes (16x16x32 bf16, 16x16x4 and 4x4x1 f32) and a vector
# instruction that reads or overwrites its result
MFMA_WAIT = 11


def registers(operand):
    m = re.fullmatch(r"v\[(\d+):(\d+)\]", operand)
    if m:
        return range(int(m.group(1)), int(m.group(2)) + 1)
    m = re.fullmatch(r"v(\d+)", operand)
    return range(int(m.group(1)), int(m.group(1)) + 1) if m else ()


def swaps_too_early(listing):
    """(number of lane swaps, those that come within MFMA_WAIT wait states of the matrix instruction that wrote one of
    their registers, along the straight line of the listing)"""
    swaps, early = 0, []
    clock, written = 0, {}
    for line in listing.splitlines():
        if line.endswith(">:"):
            clock, written = 0, {}
            name = line
        m = re.match(r"\s+([a-z]\w+)(?:\s+(.*?))?\s*(?://.*)?$", line)
        if not m:
            continue
        op, operands = m.group(1), [o.strip() for o in (m.group(2) or "").split(",")]
        if op == "s_nop":
            clock += int(operands[0], 0) + 1
            continue
        if op.startswith("v_permlane"):
            swaps += 1
            for r in (r for o in operands for r in registers(o)):
                if clock - written.get(r, -MFMA_WAIT) < MFMA_WAIT:
                    early.append((name, line.strip()))
        clock += 1
        for r in registers(operands[0]):
            written.pop(r, None)
            if op.startswith("v_mfma"):
                written[r] = clock
    return swaps, early


def test_the_check_sees_a_swap_behind_a_matrix_instruction():
    code = "0000 <k>:\n\tv_mfma_f32_16x16x32_bf16 v[4:7], v[0:3], v[8:11], v[4:7]  // 0\n%s\tv_permlane32_swap_b32_e32 v20, v6\n"
    assert len(swaps_too_early(code % "")[1]) == 1
    assert len(swaps_too_early(code % "\ts_nop 7\n\ts_nop 1\n")[1]) == 1
    assert swaps_too_early(code % "\ts_nop 10\n") == (1, [])
    assert swaps_too_early(code % "\tv_add_f32_e32 v6, v6, v6\n") == (1, [])  # (the compiler waits for that one)


@pytest.mark.parametrize("name", ["bnn_hmc_kernel", "bnn_hmc_kernel_wide"])
def test_lane_swaps_wait_for_the_matrix_instructions(lib, tmp_path, name):
    fat, co = str(tmp_path / "fat"), str(tmp_path / "co")
    subprocess.run([os.path.join(LLVM, "llvm-objcopy"), "--dump-section", ".hip_fatbin=" + fat,
                    os.path.join(BUILD, name + ".o"), str(tmp_path / "o")], check=True)
    subprocess.run([os.path.join(LLVM, "clang-offload-bundler"), "--unbundle", "--type=o", "--input=" + fat,
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--output=" + co], check=True)
    listing = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn", co], check=True,
                             stdout=subprocess.PIPE, text=True).stdout
    swaps, early = swaps_too_early(listing)
    assert swaps > 0 and not early, early[:5]
