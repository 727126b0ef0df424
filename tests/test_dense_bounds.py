"""The dense kernels' buffer resources over x end at the end of its last row, also where x is columns
of a wider matrix: they prefetch columns past the last one, and what lies past the last row need not
be the caller's memory.  Checked on the CPU: the resource's length, compiled from the kernels' own
header, and that every resource over x has it."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "crucible-strix-halo_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

# rows, ld, I, bytes per element
VIEWS = [(64, 2176, 2048, 2), (64, 2048, 2048, 4), (1, 4096, 64, 4), (16, 72, 64, 2), (0, 64, 64, 2), (64, 1 << 23, 96, 4), (8192, 2176, 2048, 2)]


def test_resource_ends_at_the_last_row(tmp_path):
    if not Path(HIPCC).exists():
        pytest.skip("no hipcc")
    src = tmp_path / "rows_bytes.hip"
    prints = "\n".join(f'  std::printf("%u\\n", cx::RowsBytes({r}, {ld}, {i}, {e}));' for r, ld, i, e in VIEWS)
    src.write_text(f'#include <cstdio>\n#include "{CSRC}/common.hpp"\nint main() {{\n{prints}\n}}\n')
    exe = tmp_path / "rows_bytes"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-std=c++20", str(src), "-o", str(exe)], check=True,
                   capture_output=True)
    got = [int(v) for v in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]
    # The end of the last element of a rows x I view with row stride ld.
    assert got == [((r - 1) * ld + i) * e if r else 0 for r, ld, i, e in VIEWS]


def test_every_resource_over_x_uses_it():
    text = (CSRC / "dense.hip").read_text()
    rsrc = re.findall(r"\brx =\s*MakeRsrc(?:Words)?\(.*?;", text, re.S)
    assert len(rsrc) == 3  # the three MFMA kernels
    assert all(re.search(r"RowsBytes\(\w+, ldx, I, esz\)", r) for r in rsrc), rsrc
