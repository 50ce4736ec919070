"""The device code the build ships, compiled with the build's own flags and disassembled (CPU):
scalar memory instructions read and nothing else, and no packed FP32 arithmetic."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
SMEM = 0b110000          # the encoding of scalar memory instructions, bits 26 to 31
READS = re.compile(r"s_(buffer_)?load_dword(x2|x4|x8|x16)?$|s_memtime$|s_memrealtime$")


@pytest.fixture(scope="module")
def instructions(tmp_path_factory):
    """(mnemonic, first word of the encoding) of every instruction."""
    from uclchem_amd import build
    if not (os.path.exists(build.HIPCC) and os.path.exists(OBJDUMP)):
        pytest.skip("no ROCm compiler")
    obj = str(tmp_path_factory.mktemp("device") / "device.o")
    flags = [f for f in build.FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([build.HIPCC, *flags, "--cuda-device-only", "--no-gpu-bundle-output", "-c", "-o", obj,
                    os.path.join(ROOT, "uclchem_amd", "csrc", "ucg_api.hip")], check=True, capture_output=True)
    text = subprocess.run([OBJDUMP, "-d", obj], check=True, capture_output=True, text=True).stdout
    found = re.findall(r"^\s+([a-z]\w+)\b.*// [0-9A-F]+: ([0-9A-F]{8})", text, re.M)
    assert len(found) > 10000
    return [(m, int(w, 16)) for m, w in found]


def test_scalar_memory_is_only_read(instructions):
    scalar = {m for m, w in instructions if w >> 26 == SMEM}
    assert any(m.startswith("s_load_dword") for m in scalar)      # the encoding is the right one
    assert all(READS.match(m) for m in scalar), sorted(scalar)


def test_no_packed_fp32_arithmetic(instructions):
    assert not {m for m, _ in instructions if re.match(r"v_pk_\w+_f32", m) and m != "v_pk_mov_f32"}
