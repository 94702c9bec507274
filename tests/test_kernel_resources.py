"""What the built kernels' code objects say about themselves (register counts,
spills, which objects hold them), where a change of the source has moved them
without changing any result."""

import os
import re
import shutil
import struct
import subprocess

import pytest

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """[(mangled name, {vgpr_count, vgpr_spill_count, ...})], one per kernel and code object."""
    from ttt_amd import _lib
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    data = open(_lib.LIB_PATH, "rb").read()
    elf = tmp_path_factory.mktemp("co") / "co.elf"
    found, at = [], data.find(MAGIC)
    while at >= 0:
        pos = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            off, size, n = struct.unpack_from("<QQQ", data, pos)
            if b"gfx950" in data[pos + 24:pos + 24 + n]:
                elf.write_bytes(data[at + off:at + off + size])
                notes = subprocess.run([READELF, "--notes", str(elf)], check=True, capture_output=True, text=True).stdout
                for k in notes.split(".group_segment_fixed_size:")[1:]:
                    found.append((re.search(r"\.name:\s+(\S+)", k)[1],
                                  {m[1]: int(m[2]) for m in re.finditer(r"\.(\w+_count):\s+(\d+)", k)}))
            pos += 24 + n
        at = data.find(MAGIC, at + 1)
    assert found
    return found


@pytest.mark.parametrize("T,F_,FF,vgprs,spilled", [
    ("DF16b", 64, 256, 256, 0), ("DF16_", 64, 256, 256, 3), ("f", 64, 256, 256, 35),
    ("DF16b", 32, 64, 128, 0), ("DF16_", 32, 64, 128, 0),  # (past 128: three waves per SIMD)
])
def test_combiner_without_kept_rows(kernels, T, F_, FF, vgprs, spilled):
    """The memory-cache combiner of an inference call (converting, two tiles per
    wave) pays no register for the rows that a training call keeps."""
    name = f"memo_combine_kernelI{T}Li{F_ // 16}ELi{FF // 16}ELNS_8MemoPassE0ELb0ELi2E"
    (k,) = [r for n, r in kernels if name in n]
    assert k["vgpr_count"] <= vgprs and k["vgpr_spill_count"] <= spilled


@pytest.mark.parametrize("kernel", ["wave16_fwd_state_kernel", "wave16_bwd_state_kernel"])
def test_fp32_kernels_in_the_fp32_object_alone(kernels, kernel):
    names = [n for n, _ in kernels if kernel in n]
    assert names and len(names) == len(set(names))
