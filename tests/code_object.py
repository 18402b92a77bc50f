"""Kernel metadata of the built library's gfx950 code object (CPU only)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "netrax_amd", "libnetrax_gpu.so")
LLVM = "/opt/rocm/llvm/bin"


def kernels(directory, *fields):
    """{mangled kernel name: {field: int}}; skips the test without the library
    or the tools."""
    objcopy = shutil.which("objcopy")
    bundler, readelf = os.path.join(LLVM, "clang-offload-bundler"), os.path.join(LLVM, "llvm-readelf")
    if not os.path.exists(LIB) or objcopy is None or not (os.path.exists(bundler) and os.path.exists(readelf)):
        pytest.skip("the HIP library, objcopy or the ROCm LLVM tools are not available")
    fat, co = str(directory / "fatbin.bin"), str(directory / "gfx950.co")
    subprocess.run([objcopy, "--dump-section", f".hip_fatbin={fat}", LIB, str(directory / "lib.so")], check=True)
    subprocess.run([bundler, "--unbundle", "--type=o", f"--input={fat}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={co}"], check=True)
    notes = subprocess.run([readelf, "--notes", co], check=True, capture_output=True, text=True).stdout
    out = {}
    for entry in re.split(r"\n  - \.", notes):
        name = re.search(r"\n\s+\.name:\s+(\S+)", "\n" + entry)
        if name:
            found = {f: re.search(r"(?:^|\n)\s*\.?" + f + r":\s+(\d+)", entry) for f in fields}
            out[name.group(1)] = {f: int(m.group(1)) for f, m in found.items() if m}
    assert out, "no kernel metadata found in the code object"
    return out
