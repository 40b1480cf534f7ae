"""Scratch memory of the built kernels, from the metadata of the library's own code objects: a read from scratch waits for every load in
flight, so in a K loop it costs up to 5 % (8192x4608x2064 in 4 groups 84.2 us, 88.4 with the lane parts of the loads there). Nothing but
256x256 tiles, whose accumulators fill the registers, may use any: up to 20 bytes outside their loops, 136 where they store partial sums.
(Without the hint on the rare kind of store those with a K tail take 28 to 32, in the loop.) No device needed."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from tritonbench_amd import _lib, build

LLVM = os.path.join(os.path.dirname(os.path.realpath(build.find_hipcc())), "..", "lib", "llvm", "bin")


def _tool(name):
    path = shutil.which(name, path=os.pathsep.join((LLVM, "/opt/rocm/llvm/bin")))
    if path is None:
        pytest.skip(f"{name} is not there")
    return path


def _code_objects(library, tmp_path):
    fat = tmp_path / "fat.bin"
    subprocess.run([_tool("llvm-objcopy"), "--dump-section", f".hip_fatbin={fat}", library, os.devnull], check=True)
    data, magic = fat.read_bytes(), b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        entry = at + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", data, at + len(magic))[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            target = data[entry + 24 : entry + 24 + length]
            entry += 24 + length
            if target.endswith(b"gfx950"):
                yield data[at + offset : at + offset + size]
        at = data.find(magic, at + 1)


def test_no_kernel_takes_scratch_into_its_loop(tmp_path):
    _lib.load()
    scratch = {}
    for i, code in enumerate(_code_objects(build.LIB_PATH, tmp_path)):
        path = tmp_path / f"{i}.co"
        path.write_bytes(code)
        notes = subprocess.run([_tool("llvm-readelf"), "--notes", str(path)], check=True, capture_output=True, text=True).stdout
        for kernel in notes.split(".agpr_count:")[1:]:
            name, size = (re.search(rf"\.{field}:\s+(\S+)", kernel).group(1) for field in ("name", "private_segment_fixed_size"))
            scratch[name] = int(size)
    assert len(scratch) > 200
    for name, size in scratch.items():
        # (the tile, its waves, whether it has a K tail, and the epilogue: plain, bias, partial sums)
        tile = re.search(r"gemm_tiled_kernelILi256ELi256ELi2ELi2ELb[01]ELi([012])E", name)
        allowed = 0 if tile is None else 136 if tile.group(1) == "2" else 20
        assert size <= allowed, f"{name}: {size} bytes of scratch"
