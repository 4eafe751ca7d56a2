"""What the compiler makes of k_rescue, read from the built library.

The kernel goes through two long phases in turn, and its lanes carry their
numbers and items from one to the other.  A function call among lanes that are
partly off, or vector registers written in lanes that are off (the compiler
does that to save its spilled scalars), has cost such lanes their values: the
band solve then read and wrote at wild addresses.  Neither may be in it."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from aeroapps_amd._lib import LIB_PATH

LLVM = "/opt/rocm/llvm/bin"
pytestmark = pytest.mark.skipif(
    not (os.path.exists(LIB_PATH) and os.path.exists(f"{LLVM}/llvm-objdump") and shutil.which("objcopy")),
    reason="library not built, or no disassembler")


def code_objects(path, tmp):
    """The gfx950 code objects of a library, one for each source file."""
    fat = os.path.join(tmp, "fatbin")
    subprocess.run(["objcopy", "-O", "binary", "--only-section=.hip_fatbin", path, fat], check=True)
    data = open(fat, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + 24)
        pos = at + 32
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", data, pos)
            target = data[pos + 24:pos + 24 + name]
            pos += 24 + name
            if target.endswith(b"gfx950") and size:
                yield data[at + offset:at + offset + size]
        at = data.find(magic, at + 24)


def test_no_calls_and_no_writes_to_lanes_that_are_off(tmp_path):
    seen = 0
    for code in code_objects(LIB_PATH, str(tmp_path)):
        if b"k_rescue" not in code:
            continue
        obj = tmp_path / "code.o"
        obj.write_bytes(code)
        names = re.findall(r"_Z\w*k_rescue\w*", subprocess.run([f"{LLVM}/llvm-readelf", "-s", "-W", str(obj)],
                                                               capture_output=True, text=True, check=True).stdout)
        names = [n for n in sorted(set(names)) if not n.endswith("kd")]
        text = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn",
                               "--disassemble-symbols=" + ",".join(names), str(obj)],
                              capture_output=True, text=True, check=True).stdout
        for body in re.split(r"^[0-9a-f]+ <(?=_Z)", text, flags=re.M)[1:]:
            seen += 1
            assert "s_swappc" not in body, body[:90]
            all_lanes = False
            for line in body.splitlines():
                ins = line.split("//")[0].strip()
                if re.match(r"s_or_saveexec_b64 s\[\d+:\d+\], -1", ins):
                    all_lanes = True
                elif all_lanes and re.match(r"s_mov_b64 exec,", ins):
                    all_lanes = False
                elif all_lanes:
                    assert not re.match(r"(v_|scratch_load|ds_|global_load|flat_load)", ins), (body[:90], ins)
    # FP64: 15 stream counts with one Stokes component and 5 with three; mixed: 7 and 2
    assert seen == 15 + 5 + 7 + 2
