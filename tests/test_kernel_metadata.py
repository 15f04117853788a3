"""The built library's kernels, from the metadata of their code objects."""
import os
import re
import struct
import subprocess

import pytest

from sgpp_amd import build

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """mangled name -> {metadata key: value} of every gfx950 kernel"""
    with open(build.LIB, "rb") as f:
        data = f.read()
    tmp, found, at = tmp_path_factory.mktemp("code"), {}, data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + n].decode()
            p += 24 + n
            if build.ARCH in name and size:
                path = str(tmp / "code_object")
                with open(path, "wb") as f:
                    f.write(data[at + offset:at + offset + size])
                notes = subprocess.run([os.path.join(build.ROCM, "llvm", "bin", "llvm-readelf"), "--notes", path],
                                       check=True, capture_output=True, text=True).stdout
                for k in re.split(r"\n  - \.a", notes)[1:]:
                    v = dict(re.findall(r"\.(\w+): +(\S+)", k))
                    found[v["name"]] = v
        at = data.find(MAGIC, at + 1)
    return found


def tree_kernels(kernels):
    """(metadata, kernel, type, register dimensions, points per lane, ModLinear, depth) of the walks"""
    out = []
    for name, v in kernels.items():
        m = re.search(r"(tree_mult\w?_kernel)I([fd])Li(\d+)ELi(\d+)ELb(\d)ELi(\d+)", name)
        if m:
            out.append((v, m[1], m[2]) + tuple(int(m[i]) for i in range(3, 7)))
    return out


def test_walks_keep_their_registers(kernels):
    """Scratch memory of the walks: a dozen registers at most (a spilled coordinate or product is
    read back at every node; two dozen made the d=10 Linear multTranspose 1.3 to 2.6 times slower)."""
    walks = tree_kernels(kernels)
    assert len(walks) >= 64
    for v, *which in walks:
        assert int(v["private_segment_fixed_size"]) <= 48, which


def test_walks_have_no_fixed_lds(kernels):
    """The walks read LDS at byte offsets from address 0, where their dynamic LDS begins as long
    as they declare no other."""
    for v, *which in tree_kernels(kernels):
        assert int(v["group_segment_fixed_size"]) == 0, which
