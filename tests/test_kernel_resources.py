"""The compiled step kernels' resources, from the metadata of the built library."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib", "llvm", "bin", "llvm-readelf")


def kernels(tmp_path):
    """{mangled name: (registers, scratch bytes, code object)} of the gfx950 code objects."""
    lib = os.path.join(ROOT, "ibtfo_amd", "libibtfo_amd.so")
    tool = READELF if os.path.isfile(READELF) else shutil.which("llvm-readelf")
    if not os.path.isfile(lib) or tool is None:
        pytest.skip("no built library or no llvm-readelf")
    data = open(lib, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    out = {}
    at = data.find(magic)
    while at >= 0:
        entry = at + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", data, at + len(magic))[0]):
            off, size, n = struct.unpack_from("<QQQ", data, entry)
            triple = data[entry + 24:entry + 24 + n].decode()
            entry += 24 + n
            if "gfx950" not in triple or size == 0:
                continue
            obj = tmp_path / "object"
            obj.write_bytes(data[at + off:at + off + size])
            notes = subprocess.run([tool, "--notes", str(obj)], capture_output=True, text=True, check=True).stdout
            for block in re.split(r"\n\s+- \.agpr_count", notes)[1:]:
                field = {k: re.search(r"\.%s:\s+(\S+)" % k, block).group(1)
                         for k in ("name", "vgpr_count", "private_segment_fixed_size")}
                out[field["name"]] = (int(field["vgpr_count"]), int(field["private_segment_fixed_size"]), at)
        at = data.find(magic, at + 1)
    return out


def test_mixed_precision_strips_hold_no_scratch(tmp_path):
    """Every mixed-precision marching strip keeps its row loop in registers (scratch
    there cost the MUSCL-Hancock form what its fourth wave per SIMD gave)."""
    strips = {n: r for n, r in kernels(tmp_path).items()
              if re.search(r"k_step(_batch|_periodic)?ILi\d+ELi\d+ELi\d+Ef", n)}
    # 3 schemes x 3 solvers x 3 limiters, each plain, with cut cells, periodic and batched
    assert len(strips) == 108
    assert {n: r for n, r in strips.items() if r[1]} == {}


def test_step_kernels_load_with_their_scheme_and_solver(tmp_path):
    """A solve loads one scheme's and solver's step kernels and none of the others': a
    code object of step kernels holds one pair, and the other kernels lie elsewhere (all
    pairs in one object cost a process's first solve 14 ms)."""
    pairs = {}
    other = set()
    for name, (_, _, obj) in kernels(tmp_path).items():
        m = re.search(r"k_(step|step_batch|step_periodic|step_rowpar|persist)ILi(\d+)ELi(\d+)E", name)
        if m:
            pairs.setdefault(obj, set()).add(m.groups()[1:])
        else:
            other.add(obj)
    assert len(pairs) == 18 and all(len(p) == 1 for p in pairs.values())
    assert not other & set(pairs)
