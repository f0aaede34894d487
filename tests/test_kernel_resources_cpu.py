"""What the compiler made of kernels whose speed depends on it, from the metadata of the
built library's code objects: an array that stays in memory (an element chosen by a
run-time index, a load from a selected address) shows as LDS or scratch that the source
does not ask for."""
import os
import re
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "k-optimizers_amd", "kaon_amd", "libkaon_amd.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    """The gfx950 code objects of the library's offload bundles."""
    at = blob.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", blob, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, pos)
            name = blob[pos + 24:pos + 24 + idlen]
            pos += 24 + idlen
            if b"gfx950" in name and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, pos)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled kernel name: (LDS bytes, scratch bytes)}"""
    if not os.path.exists(READELF) or not os.path.exists(LIB):
        pytest.skip("needs the built library and ROCm's llvm-readelf")
    with open(LIB, "rb") as fh:
        blob = fh.read()
    out = {}
    d = tmp_path_factory.mktemp("co")
    for i, co in enumerate(_code_objects(blob)):
        path = d / f"{i}.elf"
        path.write_bytes(co)
        notes = subprocess.run([READELF, "--notes", str(path)], check=True, capture_output=True, text=True).stdout
        for k in re.split(r"\n\s+- \.(?=a(?:gpr_count|rgs):)", notes)[1:]:
            name = re.search(r"\.name:\s+(_Z\w+)", k)
            if name:
                out[name.group(1)] = tuple(int(re.search(rf"\.{f}_segment_fixed_size:\s+(\d+)", k).group(1))
                                           for f in ("group", "private"))
    assert out, "no code object found in the library"
    return out


def test_kprodigy_apply_keeps_its_noise_words_in_registers(kernels):
    """k_pd2: the cautious count's four words of LDS and nothing else."""
    pd2 = {k: v for k, v in kernels.items() if "k_pd2" in k}
    assert len(pd2) >= 20
    bad = {k: v for k, v in pd2.items() if v[0] > 16 or v[1] > 0}
    assert not bad, bad
