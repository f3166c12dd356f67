"""Registers of the built population kernels: none is spilled to memory (the
batched ones run at six waves per SIMD, 80 registers, and lose more by a spill
than shorter arithmetic gives), read from the library's own code objects."""

import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "gsbn_amd", "libgsbn_amd.so")
READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    """The gfx950 entries of the offload bundles in `data`."""
    at = data.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + length]
            p += 24 + length
            if b"gfx950" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 1)


@pytest.mark.skipif(not os.path.exists(LIB) or not os.path.exists(READELF) or
                    shutil.which("c++filt") is None, reason="no built library or tools")
def test_population_kernels_spill_nothing(tmp_path):
    with open(LIB, "rb") as f:
        data = f.read()
    seen = {}
    for i, obj in enumerate(_code_objects(data)):
        p = tmp_path / ("%d.co" % i)
        p.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(p)], check=True, stdout=subprocess.PIPE,
                               text=True).stdout
        for k in re.split(r"\n\s+- \.agpr_count:", notes)[1:]:
            name = re.search(r"\.name:\s+(\S+)", k).group(1)
            name = subprocess.run(["c++filt", name], check=True, stdout=subprocess.PIPE,
                                  text=True).stdout.strip().replace("(anonymous namespace)::", "")
            seen[name.split("(")[0]] = (int(re.search(r"\.vgpr_spill_count:\s+(\d+)", k).group(1)),
                                        int(re.search(r"\.private_segment_fixed_size:\s+(\d+)",
                                                      k).group(1)))
    pop = {n: v for n, v in seen.items()
           if re.search(r"\b(pop_kernel|pop_kernel_batch|pop_kernel_batch_wave|chained_kernel|"
                        r"step_kernel|step_kernel_batch)\b", n)}
    assert len(pop) >= 13 and any("pop_kernel_batch_wave<2>" in n for n in pop)
    assert not {n: v for n, v in pop.items() if v != (0, 0)}
