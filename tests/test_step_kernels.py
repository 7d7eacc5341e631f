"""Resources of the step kernels in the built library: no scratch memory and no
spilled vector registers, which every phase's loads would wait behind."""
from __future__ import annotations

import pathlib
import re
import struct
import subprocess

import pytest

LIB = pathlib.Path(__file__).resolve().parents[1] / "leo_amd" / "_lib" / "libleo_hip.so"
READELF = pathlib.Path("/opt/rocm/llvm/bin/llvm-readelf")
KERNELS = ("leo_lane_steps", "leo_lane_steps_profiled", "leo_lane_steps_frozen")


def _code_objects(data: bytes):
    """The gfx950 code objects of the library's offload bundles (magic, count,
    then offset, size and target id of each entry)."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    for found in re.finditer(magic, data):
        start = found.start()
        at = start + len(magic)
        (count,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            target = data[at + 24:at + 24 + length]
            at += 24 + length
            if target.endswith(b"gfx950") and size:
                yield data[start + offset:start + offset + size]


def test_step_kernels_need_no_scratch(tmp_path):
    if not LIB.exists() or not READELF.exists():
        pytest.skip("needs the built library and llvm-readelf")
    seen = {}
    for i, code in enumerate(_code_objects(LIB.read_bytes())):
        path = tmp_path / f"{i}.co"
        path.write_bytes(code)
        notes = subprocess.run([str(READELF), "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"\n\s*- \.agpr_count", notes)[1:]:
            name = re.search(r"\.name:\s*(\S+)", kernel).group(1)
            short = next((k for k in KERNELS if re.fullmatch(rf"_ZN3leo{len(k)}{k}E.*", name)), None)
            if short:
                seen[short] = tuple(int(re.search(rf"\.{key}:\s*(\d+)", kernel).group(1))
                                    for key in ("private_segment_fixed_size", "vgpr_spill_count"))
    assert seen == {k: (0, 0) for k in KERNELS}
