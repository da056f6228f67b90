"""Registers and scratch of kernels whose speed rests on them, from the metadata
of the built engine's code objects."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tbtk_amd", "lib", "libtbtkx.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel name: {key: value}} of every gfx950 kernel in the library."""
    if not os.path.exists(LIB) or not os.path.exists(READELF):
        pytest.skip("needs the built engine and llvm-readelf")
    data = open(LIB, "rb").read()
    out, at = {}, data.find(MAGIC)
    path = str(tmp_path_factory.mktemp("co") / "kernels.co")
    while at >= 0:
        n, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + idlen].decode()
            p += 24 + idlen
            if not target.endswith("gfx950") or size == 0:
                continue
            with open(path, "wb") as f:
                f.write(data[at + off:at + off + size])
            notes = subprocess.run([READELF, "--notes", path], capture_output=True, text=True,
                                   check=True).stdout
            for k in re.split(r"\n  - \.", notes)[1:]:
                name = re.search(r"\.name:\s+(\S+)", k)
                if name:
                    out[name.group(1)] = {x: int(v) for x, v in re.findall(
                        r"\.(vgpr_count|private_segment_fixed_size):\s+(\d+)", k)}
        at = data.find(MAGIC, p)
    assert out
    return out


def test_gathered_batch_steps(kernels):
    """The uneven batch's step without dots: four wavefronts per SIMD (128 VGPRs)
    up to 7 slots per row, and no scratch."""
    seen = 0
    for name, k in kernels.items():
        m = re.search(r"multi_stepILi(\d)ELb\dELb0ELb\d", name)
        if m:
            seen += 1
            assert k["private_segment_fixed_size"] == 0, name
            assert k["vgpr_count"] <= (128 if int(m.group(1)) < 8 else 168), (name, k)
    assert seen == 20
