"""What the built kernels need, read from the metadata of the code objects in the core library."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from mini_engine_amd.kernels import build

_TOOLS = os.pathsep.join(("/opt/rocm/llvm/bin", os.environ.get("PATH", "")))
READELF, OBJDUMP = (shutil.which(tool, path=_TOOLS) for tool in ("llvm-readelf", "llvm-objdump"))


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


def _needs(tmp_path, kernel_name: str, *fields) -> dict:
    """Of each built kernel whose name holds `kernel_name`: the numbers of its metadata."""
    library = os.path.join(build.PKG_LIB, "libme_core.so")
    if not os.path.exists(library):
        pytest.skip("the core library is not built")
    found = {}
    for i, code in enumerate(_code_objects(open(library, "rb").read())):
        if kernel_name.encode() not in code:
            continue
        path = tmp_path / f"{i}.elf"
        path.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for kernel in notes.split("- .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel).group(1)
            if kernel_name in name:
                found[name] = tuple(int(re.search(rf"\.{field}:\s+(\d+)", kernel).group(1)) for field in fields)
    return found


@pytest.mark.skipif(READELF is None, reason="no llvm-readelf")
def test_the_decay_walk_keeps_to_its_registers(tmp_path):
    """Only the form whose lanes hold 64 rows spills, and no more than the rows that its registers cannot hold beside a batch (40);
    of waves of up to 128 rows with 16 lanes to a column two run on a SIMD, of up to 64 three."""
    seen = {}
    for name, needs in _needs(tmp_path, "decay_walk_kernel", "vgpr_spill_count", "vgpr_count").items():
        rows, lanes, rule, waves = (int(n) for n in re.findall(r"Li(\d+)E", name))
        seen[name] = (rows, lanes)
        assert needs[0] <= (40 if rows // lanes > 32 else 0), (name, needs)
        assert lanes != 16 or rows > 128 or needs[1] <= (256 if rows > 64 else 168), (name, needs)
    assert set(seen.values()) == {(rows, lanes) for rows in (32, 64, 128, 256) for lanes in (4, 16)}


@pytest.mark.skipif(READELF is None, reason="no llvm-readelf")
def test_the_recurrence_for_short_requests_leaves_room_for_three_waves(tmp_path):
    """A lane with one column of up to 64 rows: 168 registers or fewer. No form keeps anything in memory."""
    seen = set()
    for name, needs in _needs(tmp_path, "recurrence_kernelI", "private_segment_fixed_size", "vgpr_count").items():
        rows, which, heads, blocks, piece = (int(n) for n in re.findall(r"Li(\d+)E", name))
        assert needs[0] == 0, name
        if piece == 1 and heads == blocks == 1:
            seen.add(rows)
            assert needs[1] <= 168, (name, needs)
    assert seen == {16, 32, 48, 64}


def _late_reads(code: list) -> dict:
    """The most LDS reads that can be on their way at each barrier although another barrier lies between, over all paths. `code`:
    (address, name, operands, the address a branch goes to or None); reads come back in the order in which they were asked for."""
    place = {address: i for i, (address, *_) in enumerate(code)}
    most, todo, late = {0: (0, 0)}, [0], {}                     # reads from before the last barrier, reads since
    while todo:
        i = todo.pop()
        _, name, operands, target = code[i]
        old, new = most[i]
        if name.startswith("ds_read"):
            new = min(new + 1, 99)
        elif name == "s_waitcnt" and (m := re.search(r"lgkmcnt\((\d+)\)", operands)):
            new = min(new, int(m.group(1)))
            old = min(old, int(m.group(1)) - new)
        elif name == "s_barrier":
            late[i] = max(late.get(i, 0), old)
            old, new = min(old + new, 99), 0
        after = [] if name == "s_endpgm" else [i + 1]
        if target is not None:
            after = [place[target]] + (after if name.startswith("s_cbranch") else [])
        for j in after:
            was = most.get(j, (-1, -1))
            now = (max(was[0], old), max(was[1], new))
            if j < len(code) and now != was:
                most[j] = now
                todo.append(j)
    return late


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
def test_tile_products_read_lds_before_others_may_write_it(tmp_path):
    """What a wave of the tile product's kernels reads a quarter ahead is in registers before another wave can ask for the load that
    writes over it: with eight waves, of which half run later than the others, before the next barrier in front of a quarter's products
    (one that raises the wave's priority behind itself), with four before the next barrier."""
    library = os.path.join(build.PKG_LIB, "libme_core.so")
    if not os.path.exists(library):
        pytest.skip("the core library is not built")
    kernels = barriers = 0
    for i, blob in enumerate(_code_objects(open(library, "rb").read())):
        if b"gemm_tile_kernel" not in blob:
            continue
        path = tmp_path / f"{i}.elf"
        path.write_bytes(blob)
        text = subprocess.run([OBJDUMP, "-d", str(path)], capture_output=True, text=True, check=True).stdout
        pieces = re.split(r"^[0-9a-f]+ <(\S*gemm_tile_kernel\S*)>:$", text, flags=re.M)[1:]
        for name, part in zip(pieces[::2], pieces[1::2]):
            kernels += 1
            code = []
            for line in part.splitlines():
                if m := re.match(r"\s+(\w+)(.*?)\s*// ([0-9A-F]+):.*?(?:<\S+?\+0x([0-9a-f]+)>)?$", line):
                    code.append((int(m.group(3), 16), m.group(1), m.group(2), m.group(4)))
            code = [(a, name, ops, code[0][0] + int(to, 16) if to and name.startswith(("s_branch", "s_cbranch")) else None) for a, name, ops, to in code]
            waves = int(re.search(r"ILi(\d+)ELi(\d+)E", name).group(1)) * int(re.search(r"ILi(\d+)ELi(\d+)E", name).group(2))
            for j, late in _late_reads(code).items():
                if waves == 4 or (code[j + 1][1] == "s_setprio" and int(code[j + 1][2]) == 1):
                    barriers += 1
                    assert late == 0, (name, hex(code[j][0]), late)
    assert kernels == 30 and barriers >= kernels * 12        # 12 quarters in the code of a kernel
