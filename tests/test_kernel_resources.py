"""What the built kernels need, read from the metadata of the code objects in the core library."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from mini_engine_amd.kernels import build

READELF = shutil.which("llvm-readelf", path=os.pathsep.join(("/opt/rocm/llvm/bin", os.environ.get("PATH", ""))))


def _code_objects(blob: bytes):
    """The gfx950 code objects of a library's offload bundles: a magic, a count, then per entry offset, size and name."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := blob.find(magic, at)) >= 0:
        place = at + len(magic)
        count, = struct.unpack_from("<Q", blob, place)
        place += 8
        for _ in range(count if count < 64 else 0):
            offset, size, length = struct.unpack_from("<QQQ", blob, place)
            name = blob[place + 24:place + 24 + length]
            place += 24 + length
            if b"gfx950" in name and size:
                yield blob[at + offset:at + offset + size]
        at += len(magic)


@pytest.mark.skipif(READELF is None, reason="no llvm-readelf")
def test_float32_attention_keeps_to_its_registers(tmp_path):
    """No head size's instance spills to scratch, and each leaves two waves to a SIMD (512 registers)."""
    library = os.path.join(build.PKG_LIB, "libme_core.so")
    if not os.path.exists(library):
        pytest.skip("the core library is not built")
    seen = {}
    for i, code in enumerate(_code_objects(open(library, "rb").read())):
        if b"attn_f32_kernel" not in code:
            continue
        path = tmp_path / f"{i}.elf"
        path.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for kernel in notes.split("- .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel).group(1)
            if m := re.search(r"attn_f32_kernelILi(\d+)E", name):
                number = lambda field: int(re.search(rf"\.{field}:\s+(\d+)", kernel).group(1))
                seen[16 * int(m.group(1))] = (number("private_segment_fixed_size"), number("vgpr_count"))
    assert sorted(seen) == list(range(16, 129, 16))
    for head, (scratch, registers) in seen.items():
        assert scratch == 0 and registers <= 256, (head, scratch, registers)
