"""Kernels that keep their accumulators in registers have no scratch: a spilled
accumulator is a memory round trip in the innermost loop.  Read from the notes
of the built library's gfx950 code objects: no GPU."""
import os
import re
import shutil
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mojo-gemma4-cpu_amd",
                   "libbq.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{demangled kernel name: (scratch bytes, spilled vector registers)}"""
    if not os.path.exists(LIB) or not os.path.exists(READELF) or not shutil.which("c++filt"):
        pytest.skip("no built library or no tools to read it")
    data = open(LIB, "rb").read()
    path = tmp_path_factory.mktemp("objs") / "obj"
    found = {}
    for at in (m.start() for m in re.finditer(MAGIC, data)):
        n, p = struct.unpack_from("<Q", data, at + len(MAGIC))[0], at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" not in target or size == 0:
                continue
            path.write_bytes(data[at + off:at + off + size])
            notes = subprocess.run([READELF, "--notes", str(path)], check=True, capture_output=True,
                                   text=True).stdout
            for k in re.split(r"\n\s+- \.", notes):
                name = re.search(r"\.name:\s+(_Z\S+)", k)
                if name and ".vgpr_spill_count" in k:
                    found[name[1]] = (int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", k)[1]),
                                      int(re.search(r"\.vgpr_spill_count:\s+(\d+)", k)[1]))
    names = subprocess.run(["c++filt"], input="\n".join(found), check=True, capture_output=True,
                           text=True).stdout.split("\n")
    return {d.split("(")[0].replace("void ", "").replace("bq::", ""): v
            for d, v in zip(names, found.values())}


@pytest.mark.parametrize("kernel,instances", [("k_flash_attn", 20), ("k_flash_attn_rows", 28)])
def test_no_scratch(kernels, kernel, instances):
    mine = {n: v for n, v in kernels.items() if n.startswith(kernel + "<")}
    assert len(mine) == instances, sorted(mine)
    assert not {n: v for n, v in mine.items() if v != (0, 0)}
