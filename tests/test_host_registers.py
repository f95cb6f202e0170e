"""Registers and scratch memory of kernel instances, as the built library states them: what an instance loses there costs
resident waves or a trip through memory in every workgroup, and nothing else fails when it does."""
import os
import re
import struct
import subprocess

import pytest

from segquant_amd import _lib

LLVM = "/opt/rocm/llvm/bin"
pytestmark = pytest.mark.skipif(not (os.path.exists(_lib.LIB_PATH) and os.path.exists(f"{LLVM}/llvm-readelf")),
                                reason="needs the built library and the compiler's own tools")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Mangled name -> (vector registers, scratch bytes a lane) of every kernel in the library."""
    blob = open(_lib.LIB_PATH, "rb").read()
    path = str(tmp_path_factory.mktemp("objects") / "object")
    found = {}
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", blob):
        at, (count,) = m.end() + 8, struct.unpack_from("<Q", blob, m.end())
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", blob, at)
            name, at = blob[at + 24:at + 24 + length], at + 24 + length
            if size == 0 or b"gfx950" not in name:
                continue
            with open(path, "wb") as f:
                f.write(blob[m.start() + offset:m.start() + offset + size])
            notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", path], capture_output=True, text=True, check=True).stdout
            for kernel in notes.split("  - .agpr_count")[1:]:
                value = {k: re.search(rf"\.{k}:\s*(\S+)", kernel)[1] for k in ("name", "vgpr_count", "private_segment_fixed_size")}
                found[value["name"]] = int(value["vgpr_count"]), int(value["private_segment_fixed_size"])
    return found


def _pipe(bm, bn, wm, wn, fmt, fold, park, finish):
    flags = "".join(f"Lb{int(f)}E" for f in (False, park, finish) + (False,) * 6)
    return f"_ZN4segq16gemm_pipe_kernelILi{bm}ELi{bn}ELi{wm}ELi{wn}ELi{fmt}ELb{int(fold)}ELi2E{flags}EEvNS_10GemmParamsE"


@pytest.mark.parametrize("tile, fmt, fold, park, registers, scratch", [
    # several ranges of int8, parked: they have the low-rank branch, and nothing of its way through LDS
    ((256, 256, 4, 2), 0, True, True, 256, 556),
    ((256, 192, 4, 2), 0, True, True, 256, 140),
    ((192, 256, 2, 4), 0, True, True, 256, 132),
    ((256, 128, 4, 2), 0, True, True, 224, 0),
    # several ranges of e4m3: two workgroups share a compute unit
    ((128, 128, 4, 2), 1, True, False, 128, 0),
    # one range
    ((256, 256, 4, 2), 0, False, False, 256, 0),
    ((256, 256, 4, 2), 1, False, False, 256, 16),
    ((384, 192, 4, 2), 0, False, False, 256, 12),
    ((384, 192, 4, 2), 1, False, False, 256, 12),
])
def test_instances_that_finish_in_output_units(kernels, tile, fmt, fold, park, registers, scratch):
    vgpr, bytes_ = kernels[_pipe(*tile, fmt, fold, park, True)]
    assert vgpr <= registers and bytes_ <= scratch
