"""What the compiler made of kernels whose design stands on it, read from the libraries that are built here (no GPU)."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from pico_vllm_amd.ops import library


def kernels_of(path, tmp_path):
    """{mangled name: bytes of private memory a lane} of every kernel in a library's gfx950 code objects."""
    tool = next((t for t in (shutil.which("llvm-readelf"), "/opt/rocm/llvm/bin/llvm-readelf") if t and os.path.isfile(t)), None)
    if tool is None:
        pytest.skip("no llvm-readelf")
    with open(path, "rb") as f:
        data = f.read()
    out = {}
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        entries, at = struct.unpack_from("<Q", data, m.end())[0], m.end() + 8
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            if data[at + 24:at + 24 + length].endswith(b"gfx950"):
                obj = tmp_path / "code.elf"
                obj.write_bytes(data[m.start() + offset:m.start() + offset + size])
                notes = subprocess.run([tool, "--notes", str(obj)], capture_output=True, text=True, check=True).stdout
                out.update((n, int(b)) for n, b in re.findall(r"\.name:\s+(\S+)\n(?:(?!\.name:).)*?\.private_segment_fixed_size:\s+(\d+)", notes, re.S))
            at += 24 + length
    return out


@pytest.mark.parametrize("dk,dv", [(32, 96), (64, 128), (96, 96), (128, 96), (128, 128), (256, 224), (320, 256)])
def test_staged_keys_travel_in_registers(tmp_path, dk, dv):
    # the next keys and values are asked for under a stage's products: held in private memory they would be waited for at once
    path = library.build_library(f"pico_attnb_k{dk}_v{dv}", library.ATTN_BIAS_SOURCES, (f"-DPICO_DK={dk}", f"-DPICO_DV={dv}"))
    found = {n: b for n, b in kernels_of(path, tmp_path).items() if "attn_bias_staged_kernel" in n}
    assert len(found) == 1 and set(found.values()) == {0}, found


def test_rows_of_an_expert_are_looked_up_with_all_lanes_on(tmp_path):
    # a lane that is off while another reads it need not hold its value: an expert would be missed, or taken twice
    out = str(tmp_path / "moe_mfma.s")
    subprocess.run([library._hipcc(), *library.HIP_FLAGS, "-I", library.CSRC, "--cuda-device-only", "-S",
                    os.path.join(library.CSRC, "moe_mfma.hip"), "-o", out], check=True, capture_output=True)
    with open(out) as f:
        bodies = re.findall(r"^_Z\d+moe_(?:up|down)_rows_kernelILb1E\S*:(.*?)s_endpgm", f.read(), re.M | re.S)
    assert len(bodies) == 2
    for body in bodies:
        reads = 0
        for block in re.split(r"^\.LBB\S+:|s_or_b64 exec, exec", body, flags=re.M):       # (where lanes come back on, or another way joins)
            saved = False
            for line in block.splitlines():
                saved = saved or "saveexec" in line
                if "v_readlane" in line:
                    reads += 1
                    assert not saved, block
        assert reads
