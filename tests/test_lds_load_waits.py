"""Loads into LDS written as assembly keep the wait states that the compiler does not see to there: five between a vector
instruction that writes the scalar base (a readfirstlane, the readlane of a spilled register) and the load, one between the
write of m0 and the load.  Compiled to assembly and read, no GPU."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "salt-core_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

pytestmark = pytest.mark.skipif(not Path(HIPCC).exists(), reason="no hipcc")

# the base is made per lane and used at once: nothing but the load itself keeps its distance
NEAR = """
#include "lds_load.h"
using namespace mi355;
__global__ __launch_bounds__(64) void near_kernel(const uint8_t *const *from, uint4 *out) {
    __shared__ __attribute__((aligned(16))) uint8_t stage[1024];
    const uint32_t offset = threadIdx.x * 16u;
    const uint8_t *const p = from[threadIdx.x];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    load_to_lds<16>(uniform_address((lds_load_from)(uintptr_t)p), offset, stage);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    out[threadIdx.x] = ((const uint4 *)stage)[threadIdx.x];
}
"""


def assembly(source, tmp_path):
    out = tmp_path / "out.s"
    subprocess.check_call([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off",
                           "-fno-gpu-flush-denormals-to-zero", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                           "-w", "-I", str(CSRC), "--cuda-device-only", "-S", str(source), "-o", str(out)])
    lines = [re.split(r";|//", line)[0].strip() for line in out.read_text().splitlines()]
    return [line for line in lines if line and not line.startswith(".") and not line.endswith(":")]


def scalars(operand):
    pair = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if pair:
        return set(range(int(pair[1]), int(pair[2]) + 1))
    return {int(operand[1:])} if re.fullmatch(r"s\d+", operand) else {"m0"} if operand == "m0" else set()


def written(line):
    return scalars(line.split(None, 1)[1].split(",")[0].strip()) if " " in line else set()


def states_since_write(code, at, registers):
    """(instruction, wait states between it and code[at]) of the last writes of the registers, in program order"""
    found, left, states = [], set(registers), 0
    for line in reversed(code[max(0, at - 600):at]):
        if written(line) & left:
            found.append((line, states))
            left -= written(line)
        nop = re.match(r"s_nop (\d+)", line)
        states += int(nop[1]) + 1 if nop else 1
    return found


@pytest.mark.parametrize("source", ["near", "q4_mfma.hip", "nvfp4_mfma.hip"])
def test_loads_into_lds_keep_their_distance(source, tmp_path):
    path = CSRC / source
    if source == "near":
        path = tmp_path / "near.hip"
        path.write_text(NEAR)
    code = assembly(path, tmp_path)
    loads = [i for i, line in enumerate(code) if line.startswith("global_load_lds")]
    assert loads
    for i in loads:
        operands = [o.strip() for o in code[i].split(None, 1)[1].split(",")]
        for writer, states in states_since_write(code, i, scalars(operands[1].split()[0])):
            assert not writer.startswith("v_") or states >= 5, (writer, states, code[i])
        for writer, states in states_since_write(code, i, {"m0"}):
            assert states >= 1 and (not writer.startswith("v_") or states >= 5), (writer, states, code[i])
