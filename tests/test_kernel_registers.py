"""Registers of the built kernels, from the code objects in libsfnx_moe.so: a kernel that spills, or takes one register more
than its wavefronts a SIMD allow, computes the same values in up to twice the time, which no other test shows."""
import re
import struct
import subprocess
from pathlib import Path

import pytest

from sfnx_amd import _abi

READELF = Path("/opt/rocm/llvm/bin/llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled kernel name: (VGPRs, spilled VGPRs)}"""
    if not _abi.LIB_PATH.exists() or not READELF.exists():
        pytest.skip("the library is not built, or llvm-readelf is missing")
    lib, out = _abi.LIB_PATH.read_bytes(), {}
    obj = tmp_path_factory.mktemp("co") / "co"
    for m in re.finditer(MAGIC, lib):
        n, at = struct.unpack_from("<Q", lib, m.end())[0], m.end() + 8
        if n > 8:
            continue   # the magic as text
        for _ in range(n):
            off, size, tl = struct.unpack_from("<QQQ", lib, at)
            triple, at = lib[at + 24:at + 24 + tl], at + 24 + tl
            if b"gfx950" not in triple or not size:
                continue
            obj.write_bytes(lib[m.start() + off:m.start() + off + size])
            text = subprocess.run([READELF, "--notes", obj], capture_output=True, text=True, check=True).stdout
            for k in re.split(r"\n  - (?=\.agpr_count|\.args)", text)[1:]:
                f = {a: b for a, b in re.findall(r"\n    \.(name|vgpr_count|vgpr_spill_count): +(\S+)", k)}
                out[f["name"]] = int(f["vgpr_count"]), int(f["vgpr_spill_count"])
    assert out
    return out


def test_decode_kernels_do_not_spill(kernels):
    dec = {n: v for n, v in kernels.items() if "k_dec_" in n or "k_moe_mv" in n or "k_route" in n}
    assert len(dec) > 100
    assert not {n: v for n, v in dec.items() if v[1]}


@pytest.mark.parametrize("wtype", [2, 7, 8])
@pytest.mark.parametrize("G", [2, 4])
def test_window_gate_up_two_workgroups(kernels, wtype, G):
    """the windows' gate|up of the 32-value types up to 2048 columns: 1024-thread workgroups, two a compute unit in 64
    registers"""
    v = [v[0] for n, v in kernels.items() if f"k_dec_expertsILi{wtype}ELi{G}E" in n]
    assert v and max(v) <= 64
