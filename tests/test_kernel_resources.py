"""Registers of the one-row stage kernels whose third wave per SIMD depends on
them (168 of 512 each), from the kernel metadata of the built library; no GPU
needed."""
import os
import re
import struct
import subprocess

import pytest

from dgpr_amd import build

# template arguments P, Q, W, record type, AFF, STO
KERNELS = {
    "p = 1 affine": "ILi1ELi1ELi%dEdLb1ELb0EE",
    "p = 1 affine, FP32 records": "ILi1ELi1ELi%dEfLb1ELb0EE",
    "p = 2 affine": "ILi2ELi1ELi%dEdLb1ELb0EE",
    "p = 2 curved": "ILi2ELi1ELi%dEdLb0ELb0EE",
    "p = 3 affine": "ILi3ELi1ELi%dEdLb1ELb0EE",
    "p = 3 curved": "ILi3ELi1ELi%dEdLb0ELb0EE",
}
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    """The gfx950 code objects of the offload bundles in a library."""
    at = data.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, k = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24:p + 24 + k].decode()
            p += 24 + k
            if "gfx950" in triple and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def report(tmp_path_factory):
    if not os.path.exists(build.OUT):
        build.build()
    with open(build.OUT, "rb") as f:
        data = f.read()
    readelf = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
    out = {}
    for i, obj in enumerate(code_objects(data)):
        path = tmp_path_factory.mktemp("code") / ("%d.elf" % i)
        path.write_bytes(obj)
        notes = subprocess.run([readelf, "--notes", str(path)], capture_output=True, text=True,
                               check=True, timeout=120).stdout
        for k in notes.split("- .agpr_count:")[1:]:
            out[re.search(r"\.symbol:\s+(\S+)", k).group(1)] = (
                int(re.search(r"\.vgpr_count:\s+(\d+)", k).group(1)),
                int(re.search(r"\.vgpr_spill_count:\s+(\d+)", k).group(1)))
    return out


@pytest.mark.parametrize("waves", [2, 3])
@pytest.mark.parametrize("name", list(KERNELS))
def test_three_waves_without_spills(report, name, waves):
    tag = "dgx_rhs_stage_kernel" + KERNELS[name] % waves
    (vgprs, spilled), = [v for k, v in report.items() if tag in k]
    print(name, vgprs, "registers", spilled, "spilled")
    assert vgprs <= 168 and spilled == 0
