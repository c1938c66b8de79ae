"""Registers of the built step kernels, from the metadata of the library's own
gfx950 code objects (no GPU needed): the FP64 kernels of the time step keep
everything in registers.  FP64 holds twice the registers of FP32, so a budget
measured in FP32 does not carry over."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "lbm3_amd", "liblbm3mi.so")
LLVM = "/opt/rocm/llvm/bin/"


def _kernels(tmp_path):
    """{mangled kernel name: {metadata key: value}} over the library's code objects."""
    section = tmp_path / "fatbin"
    subprocess.run([LLVM + "llvm-objcopy", "--dump-section", ".hip_fatbin=%s" % section, LIB, "/dev/null"], check=True)
    data = section.read_bytes()
    out = {}
    # each object file brings a bundle: count, then (offset, size, triple) of each entry
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        base = m.start()
        count = int.from_bytes(data[base + 24:base + 32], "little")
        p = base + 32
        for _ in range(count):
            off, size, n = (int.from_bytes(data[p + 8 * k:p + 8 * k + 8], "little") for k in range(3))
            triple = data[p + 24:p + 24 + n]
            p += 24 + n
            if b"gfx950" not in triple:
                continue
            obj = tmp_path / "code"
            obj.write_bytes(data[base + off:base + off + size])
            notes = subprocess.run([LLVM + "llvm-readelf", "--notes", str(obj)], check=True, capture_output=True, text=True).stdout
            for block in notes.split("  - .agpr_count:")[1:]:
                keys = dict(re.findall(r"^ +(\.\w+): +(\S+)$", block, re.M))
                out[keys[".name"]] = keys
    return out


@pytest.mark.skipif(not os.path.exists(LIB), reason="the library is not built")
def test_fp64_step_kernels_do_not_spill(tmp_path):
    kernels = _kernels(tmp_path)
    fp64 = {k: v for k, v in kernels.items() if re.search(r"k_(collide_stream|collide_stream_walls|open_groups|rotor_cells)Id", k)}
    assert len(fp64) > 20
    assert any("k_collide_stream_wallsId" in k for k in fp64)
    spills = {k: int(v[".vgpr_spill_count"]) for k, v in fp64.items() if int(v[".vgpr_spill_count"])}
    assert not spills
