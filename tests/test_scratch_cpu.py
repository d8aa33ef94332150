"""Register spills of the built kernels, from the code objects' own metadata: a
scan kernel whose chunk loop spills goes through scratch memory at every step, which
no numerics test shows."""
import re
import shutil
import struct
import subprocess
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parents[1] / "gdn2-jax-kernel_amd" / "gdn2_package" / "libgdn2_hip.so"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _tool(name):
    for cand in (shutil.which(name), f"/opt/rocm/llvm/bin/{name}"):
        if cand and Path(cand).exists():
            return cand
    pytest.skip(f"{name} not found")


def _code_objects(fatbin: bytes):
    """The gfx950 entries of the offload bundles in a .hip_fatbin section."""
    at = fatbin.find(MAGIC)
    while at >= 0:
        count, o = struct.unpack_from("<Q", fatbin, at + 24)[0], at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", fatbin, o)
            if b"gfx950" in fatbin[o + 24:o + 24 + n]:
                yield fatbin[at + off:at + off + size]
            o += 24 + n
        at = fatbin.find(MAGIC, at + 24)


@pytest.fixture(scope="module")
def scratch(tmp_path_factory):
    """{mangled kernel name: scratch bytes per lane} of the built library."""
    if not LIB.exists():
        pytest.skip("library not built")
    tmp = tmp_path_factory.mktemp("co")
    subprocess.run([_tool("llvm-objcopy"), f"--dump-section=.hip_fatbin={tmp / 'fat'}", str(LIB),
                    str(tmp / "copy.so")], check=True)
    out = {}
    for i, co in enumerate(_code_objects((tmp / "fat").read_bytes())):
        (tmp / f"{i}.elf").write_bytes(co)
        notes = subprocess.run([_tool("llvm-readelf"), "--notes", str(tmp / f"{i}.elf")], check=True,
                               capture_output=True, text=True).stdout
        # a kernel's entries are in alphabetical order: its name, then its scratch size
        for name, size in re.findall(r"\.name:\s+(_ZN4gdn2\S+)\n.*?\.private_segment_fixed_size: (\d+)",
                                     notes, re.S):
            out[name] = int(size)
    return out


# mangled template arguments: fwd_scan<T, BT, D, KS, CPW, NO, SUM>
@pytest.mark.parametrize("kernels,limit", [
    (r"fwd_scanIfLi64ELi64E", 0),       # float32, D = 64: every form
    (r"fwd_scanIfLi64ELi256E", 64),     # float32, D = 256: a few addresses, spilled once
])
def test_scans_without_scratch(scratch, kernels, limit):
    found = {k: v for k, v in scratch.items() if re.search(kernels, k)}
    assert found
    assert max(found.values()) <= limit, found
