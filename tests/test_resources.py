"""Registers and LDS of the built kernels whose speed rests on two work-groups per CU, from the metadata
notes of the library's own code objects.  Needs the build and ROCm's llvm-readelf, no GPU."""
import os
import re
import struct
import subprocess

import pytest

from co_alibi_attn import _native

READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
TYPES = {"DF16_": 2, "DF16b": 2, "f": 4}


def _code_objects(data):
    """The gfx950 code objects of the offload bundles in a library."""
    at = data.find(MAGIC)
    while at >= 0:
        pos = at + len(MAGIC)
        (n,) = struct.unpack_from("<Q", data, pos)
        pos += 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24: pos + 24 + idlen]
            pos += 24 + idlen
            if b"gfx950" in name and size:
                yield data[at + off: at + off + size]
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{(kernel, element bytes, head dim): [(name, registers, LDS bytes)]} of the library."""
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    _native.lib()
    out = {}
    for i, obj in enumerate(_code_objects(open(_native.LIB_PATH, "rb").read())):
        path = tmp_path_factory.mktemp("co") / f"{i}.elf"
        path.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for entry in re.split(r"\n  - (?=\.\w)", notes):
            name = re.search(r"^\s*\.name: +(\S+)$", entry, re.M)
            vgpr = re.search(r"^\s*\.vgpr_count: +(\d+)", entry, re.M)
            lds = re.search(r"^\s*\.group_segment_fixed_size: +(\d+)", entry, re.M)
            if not (name and vgpr and lds):
                continue
            m = re.search(r"coalibi_(\w+?)_kernelI(DF16_|DF16b|f)Li(\d+)E", name.group(1))
            if m:
                key = (m.group(1), TYPES[m.group(2)], int(m.group(3)))
                out.setdefault(key, []).append((name.group(1), int(vgpr.group(1)), int(lds.group(1))))
    assert out, "no kernels parsed"
    return out


# A SIMD has 512 registers per lane: 256 for each of two wavefronts.
@pytest.mark.parametrize("kernel,size,dims", [
    ("fwd", 2, (16, 32, 64, 128)),
    ("fwd", 4, (16, 32, 64)),
    ("fwd_split", 2, (16, 32, 64, 128)),
    ("fwd_split", 4, (16, 32, 64)),
    ("bwd_dq", 2, (16, 32, 64, 128)),
    ("bwd_dq_split", 2, (16, 32, 64, 128)),
    ("bwd_dkdv_store", 2, (64, 128)),
    ("decode_split", 2, (32, 64, 128)),
], ids=str)
def test_two_work_groups_per_cu(kernels, kernel, size, dims):
    for D in dims:
        built = kernels[(kernel, size, D)]
        if (kernel, size, D) == ("fwd", 4, 64):  # also built for one per CU, for grids that give a CU one
            built = [k for k in built if "Li1EEEv" not in k[0]]
        for name, regs, lds in built:
            assert regs <= 256 and lds <= 80 * 1024, (name, regs, lds)
