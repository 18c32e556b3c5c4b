"""What the compiler reports for kernels in the built library: the StandardForm line kernels of scalar laws
keep all their values in vector registers (a bound on the registers that is too tight for a shape
makes them spill to memory, with the same results)."""

import os
import re
import shutil
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cloud.jl_amd", "csrc", "libsse_hip.so")
READELF = shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin")
EM_AMDGPU = 224


def _device_images(blob):
    """The AMDGPU ELF files inside the library, each to the end of its section headers."""
    at = blob.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", blob, at + 18)[0] == EM_AMDGPU:
            shoff, = struct.unpack_from("<Q", blob, at + 40)
            size, count = struct.unpack_from("<HH", blob, at + 58)
            yield blob[at:at + shoff + size * count]
        at = blob.find(b"\x7fELF", at + 4)


@pytest.mark.skipif(READELF is None or not os.path.exists(LIB), reason="no built library or no llvm-readelf")
def test_standard_line_kernels_do_not_spill(tmp_path):
    spills = {}
    with open(LIB, "rb") as f:
        blob = f.read()
    for n, image in enumerate(_device_images(blob)):
        path = tmp_path / f"{n}.co"
        path.write_bytes(image)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for name, count in re.findall(r"\.name:\s+(\S+).*?\.vgpr_spill_count:\s+(\d+)", notes, re.S):
            if re.match(r"_ZN3sse\d+k_std_(nodal|aux|td)_tensor", name):
                spills[name] = int(count)
    # 9 shapes: nodal values, two mappings of the gradient, four time derivatives
    assert len(spills) == 9 * 7, sorted(spills)
    assert not any(spills.values()), {k: v for k, v in spills.items() if v}
