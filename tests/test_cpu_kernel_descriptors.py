"""CPU: what the built library's kernels ask of the dispatch (their kernel descriptors)."""

from __future__ import annotations

import re
import shutil
import struct
import subprocess

import pytest

from cugo_amd import build
from tests.conftest import REPO

READELF = build.LLVM_BIN / "llvm-readelf"


def descriptors(obj) -> dict[str, bytes]:
    """The 64-byte descriptor of every kernel in a code object, by mangled name."""
    run = lambda *a: subprocess.run([str(READELF), *a, str(obj)], check=True,  # noqa: E731
                                    capture_output=True, text=True).stdout
    sections = {int(m[1]): (int(m[2], 16), int(m[3], 16)) for m in re.finditer(
        r"\[\s*(\d+)\] \S+\s+\S+\s+([0-9a-f]{16}) ([0-9a-f]+)", run("-S", "-W"))}
    data, found = obj.read_bytes(), {}
    for m in re.finditer(r"([0-9a-f]{16})\s+64 OBJECT\s+\S+\s+\S+\s+(\d+) (\S+)\.kd",
                         run("-s", "-W")):
        address, offset = sections[int(m[2])]
        at = int(m[1], 16) - address + offset
        found[m[3]] = data[at:at + 64]
    return found


def test_no_kernel_reads_the_dispatch_packet(tmp_path):
    """A kernel that reads the dispatch packet (kernel code property bit 1) waits for host
    memory in every workgroup; the compiler makes one read it to keep an array or a struct's
    padding in LDS by thread."""
    if not READELF.exists() or not shutil.which("objcopy"):
        pytest.skip("no ROCm LLVM tools")
    kernels = {}
    for obj in build.code_objects(REPO / "cugo_amd" / "libcugo_hip.so", tmp_path):
        kernels.update(descriptors(obj))
    assert len(kernels) > 100
    for name, d in kernels.items():
        properties, = struct.unpack_from("<H", d, 56)
        assert properties & 2 == 0, f"{name} reads the dispatch packet"
