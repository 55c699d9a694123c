"""What the compiler allotted to kernels of the main path, read from the metadata of the built
library's own code objects: no scratch memory and no spilled vector registers.  A periodic line
solve whose general form spilled took 8 % longer, and the convolutions whose kernel pieces went
through scratch 3 to 5 us longer per call."""
import os
import re
import shutil
import struct
import subprocess

import pytest

import simpletcsolver_amd as tc

TOOLS = "/opt/rocm/llvm/bin"


def _tool(name):
    p = os.path.join(TOOLS, name)
    return p if os.path.exists(p) else shutil.which(name)


def code_objects(path, tmp):
    """the gfx950 code objects of a library's .hip_fatbin section (a sequence of bundles: magic,
    entry count, then offset, size, id length and id of each entry)"""
    fat = os.path.join(tmp, "fat.bin")
    subprocess.run([_tool("llvm-objcopy"), "--dump-section", f".hip_fatbin={fat}", path, os.path.join(tmp, "copy.so")], check=True)
    data = open(fat, "rb").read()
    for m in re.finditer(rb"__CLANG_OFFLOAD_BUNDLE__", data):
        at = m.start()
        n, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen].decode()
            p += 24 + idlen
            if "gfx950" in name:
                yield data[at + off:at + off + size]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(tc.LIB_PATH):
        pytest.skip("the library is not built")
    if not _tool("llvm-objcopy") or not _tool("llvm-readelf"):
        pytest.skip("LLVM's binary tools are not installed")
    tmp = str(tmp_path_factory.mktemp("co"))
    out = {}
    for q, co in enumerate(code_objects(tc.LIB_PATH, tmp)):
        p = os.path.join(tmp, f"{q}.co")
        open(p, "wb").write(co)
        notes = subprocess.run([_tool("llvm-readelf"), "--notes", p], check=True, capture_output=True, text=True).stdout
        for block in re.split(r"\n\s+- \.agpr_count:", notes)[1:]:
            def field(k):
                return re.search(rf"\.{k}:\s+(\S+)", block).group(1)
            out[field("name")] = (int(field("private_segment_fixed_size")), int(field("vgpr_spill_count")))
    return out


@pytest.mark.parametrize("name,count", [("tck_cnn_conv", 3), ("tck_cnn_wgrad", 3), ("tck_psolve", 2), ("tck_pxsolve", 10)])
def test_no_scratch_and_no_spills(kernels, name, count):
    found = {k: v for k, v in kernels.items() if re.match(rf"_Z\d+{name}(I|E|P|[0-9])", k)}
    assert len(found) == count, sorted(found)
    assert all(v == (0, 0) for v in found.values()), found
