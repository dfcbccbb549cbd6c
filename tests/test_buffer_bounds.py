"""Kernels that read past the end of a sequence, block or head row as zero leave it to the
bounds check of raw buffer accesses.  That check is documented for the lane offset (and the
instruction's own); the scalar offset is left out of it.  So no buffer access of those kernels
may carry a scalar offset: read from the AMD assembly of the sources (compiled here, run
nowhere)."""
from __future__ import annotations

import pathlib
import re
import shutil
import subprocess

import pytest

PKG = pathlib.Path(__file__).resolve().parent.parent / "gguf-runner_amd"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

# operands: [data,] lane offset (or "off"), descriptor, scalar offset
ACCESS = re.compile(r"^\s*buffer_(?:load|store|atomic)_\w+\s+(?:[^,\s]+(?:\[[^\]]*\])?,\s*)+s\[\d+:\d+\],\s*(\S+)")


@pytest.mark.parametrize("source", ["deltanet.hip", "encoder.hip"])
def test_bounds_checked_accesses_have_no_scalar_offset(tmp_path, source):
    if not pathlib.Path(HIPCC).exists():
        pytest.skip("no hipcc")
    out = tmp_path / "kernels.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", f"-I{PKG.parent / 'include'}",
                    f"-I{PKG / 'csrc'}", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-w", "-S",
                    "--cuda-device-only", str(PKG / "csrc" / source), "-o", str(out)], check=True,
                   stderr=subprocess.DEVNULL)
    lines = [x for x in out.read_text().splitlines() if re.match(r"\s*buffer_(load|store|atomic)_", x)]
    assert lines
    offsets = {x.strip(): ACCESS.match(x) for x in lines}
    assert all(offsets.values()), [x for x, m in offsets.items() if not m][:3]
    assert not [x for x, m in offsets.items() if m.group(1) != "0"]
