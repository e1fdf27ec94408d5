"""What the compiler made of the kernels, from the notes in the built library's own code objects: kernels whose registers are counted keep none of them in memory."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name -> its note, of every kernel in libaxhip.so"""
    data = open(os.path.join(ROOT, "axiom_amd", "lib", "libaxhip.so"), "rb").read()
    out = {}
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at = m.start() + 32
        for _ in range(struct.unpack_from("<Q", data, m.start() + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            name, at = data[at + 24:at + 24 + length], at + 24 + length
            if b"gfx950" not in name or not size:
                continue
            path = tmp_path_factory.mktemp("code") / "code.o"
            path.write_bytes(data[m.start() + offset:m.start() + offset + size])
            notes = subprocess.run(["/opt/rocm/llvm/bin/llvm-readelf", "--notes", str(path)], capture_output=True, text=True, check=True).stdout
            for note in notes.split("  - .agpr_count")[1:]:
                out[re.search(r"\.name: +(\S+)", note).group(1)] = note
    return out


def test_planes_keep_their_registers(kernels):
    """Also with the second pass for sums that are not finite, which few products take and all of them would pay for."""
    mine = {name: note for name, note in kernels.items() if "k_gemm_planes" in name or "k_cut_planes" in name}
    assert len(mine) == 7
    for name, note in mine.items():
        assert re.search(r"\.private_segment_fixed_size: 0\n", note) and re.search(r"\.vgpr_spill_count: 0\n", note), name
