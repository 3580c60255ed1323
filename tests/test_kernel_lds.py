"""CPU tests of the built kernels' resources: the metadata of the library's gfx950
code objects states each kernel's static LDS, which has to hold what its workgroup
stages there, and how many of its vector registers live in memory."""
import os
import re
import struct
import subprocess

import pytest

from conftest import PKG

LIB = os.path.join(PKG, "lib", "libloom_infer_hip.so")
READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")


def code_objects(blob):
    """The gfx950 ELF images of the offload bundles in `blob`."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = blob.find(magic)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", blob, at + len(magic))
        p = at + len(magic) + 8
        for _ in range(n):
            off, size, width = struct.unpack_from("<QQQ", blob, p)
            triple = blob[p + 24:p + 24 + width]
            p += 24 + width
            if b"gfx950" in triple:
                yield blob[at + off:at + off + size]
        at = blob.find(magic, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Kernel symbol -> (bytes of static LDS, spilled vector registers)."""
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    out = {}
    for i, image in enumerate(code_objects(open(LIB, "rb").read())):
        path = tmp_path_factory.mktemp("co") / f"{i}.elf"
        path.write_bytes(image)
        notes = subprocess.run([READELF, "--notes", str(path)], check=True, capture_output=True,
                               text=True).stdout
        for k in re.split(r"^\s+- \.agpr_count", notes, flags=re.M)[1:]:
            name = re.search(r"^ {4}\.name:\s+(\S+)", k, flags=re.M).group(1)
            out[name] = tuple(int(re.search(r"\.%s:\s+(\d+)" % f, k).group(1))
                              for f in ("group_segment_fixed_size", "vgpr_spill_count"))
    return out


def test_pipelined_tiles_hold_their_staging(kernels):
    """After its walk each wave of a pipelined long tile stages 32 rows of O, 272
    bytes apart, beside the workgroup's column states (max and normalizer of 32
    columns and a flag per wave) and each wave's 64 page indices."""
    found = {}
    for name, (have, _) in kernels.items():
        m = re.search(r"(paged|ragged)_prefill_pipe_kernelILi(\d)ELi(\d)E(?:Lb([01])E)?", name)
        if not m:
            continue
        waves = int(m.group(2))
        need = waves * (32 * 272 + 2 * 32 * 4 + 4 + 64 * 4)
        if int(m.group(3)) < waves:  # several wave groups: the merge of their columns' states
            need = max(need, waves * (64 * 64 * 4 + 2 * 32 * 4 + 4 + 64 * 4))
        found[m.group(0)] = (have, need)
    assert len(found) == 12
    short = {k: v for k, v in found.items() if v[0] < v[1]}
    assert not short, short


def test_no_kernel_spills_vector_registers(kernels):
    """A spilled register of a tile's walk costs a memory round trip per block.
    (The plain FP8 tiles of 128 columns hold 14 in scratch: three of their
    workgroups per CU are still faster than two, on the short contexts that they
    serve.)"""
    assert len(kernels) > 50
    spilled = {k: n for k, (_, n) in kernels.items()
               if n and "paged_prefill_kernelILi4ELb1ELb1ELi2E" not in k}
    assert spilled == {}
