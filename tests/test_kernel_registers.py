"""Register spills of the built kernels, from the metadata in libdramamoe.so (CPU)."""
import re
import shutil
import subprocess

import pytest

import dramamoe as D

READELF = shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin:/opt/rocm/bin")


def _spills(tmp_path):
    """{kernel: spilled vector registers} over the gfx950 code objects embedded in the library."""
    data, out = open(D.LIB_PATH, "rb").read(), {}
    for m in re.finditer(b"\x7fELF", data):
        if data[m.start() + 18:m.start() + 20] != b"\xe0\x00":  # EM_AMDGPU
            continue
        f = tmp_path / "code.o"
        f.write_bytes(data[m.start():])
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True).stdout
        for k, n in re.findall(r"\.name:\s+(\S+)(?:(?!\.name:).)*?\.vgpr_spill_count:\s+(\d+)", notes, re.S):
            out[k] = int(n)
    return out


@pytest.mark.skipif(READELF is None, reason="no llvm-readelf")
def test_streaming_kernels_do_not_spill(tmp_path):
    """A spill is a vector memory operation: it waits for the weight loads in flight of these kernels."""
    spills = {k: n for k, n in _spills(tmp_path).items() if "k_grouped" in k or "k_gemm" in k}
    assert len(spills) > 40
    assert not {k: n for k, n in spills.items() if n}
