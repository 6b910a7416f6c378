"""Registers of the built kernels, from the metadata in the library's own code objects.  No GPU needed."""
import re
import subprocess
from pathlib import Path

import pytest

READELF = Path("/opt/rocm/llvm/bin/llvm-readelf")


def kernels(tmp_path):
    """{mangled name: spilled vector registers} of every kernel in the library."""
    from olmax_amd import _lib
    if not _lib.lib_path().exists() or not READELF.exists():
        pytest.skip("needs the built library and llvm-readelf")
    blob, out = _lib.lib_path().read_bytes(), {}
    for at in (m.start() for m in re.finditer(b"\x7fELF\x02\x01\x01\x40", blob)):  # ELFOSABI_AMDGPU_HSA
        elf = tmp_path / f"{at}.elf"
        elf.write_bytes(blob[at:])  # (a reader takes what the headers name)
        notes = subprocess.run([str(READELF), "--notes", str(elf)], capture_output=True, text=True).stdout
        elf.unlink()
        for kernel in notes.split("\n  - .agpr_count")[1:]:
            out[re.search(r"\.name: +(\S+)", kernel)[1]] = int(re.search(r"\.vgpr_spill_count: (\d+)", kernel)[1])
    return out


def test_cross_entropy_rows_stay_in_registers(tmp_path):
    got = {name: n for name, n in kernels(tmp_path).items() if "ce_row_regs_kernel" in name}
    assert len(got) >= 20
    assert not any(got.values()), {name: n for name, n in got.items() if n}
