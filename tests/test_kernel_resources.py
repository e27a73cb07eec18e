"""What the built kernels use, from the metadata of the code objects in
libsevc.so: a copy that is to have four 16-byte loads in flight a lane needs 16
registers for them, and no LDS to put them in."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from sevc.build import LIB

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"


def _code_objects():
    """The gfx950 code objects of the offload bundles (clang's format: a magic
    text, a count, then offset, size and target of each entry)."""
    data = open(LIB, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    for m in re.finditer(magic, data):
        at = m.end()
        n, = struct.unpack_from("<Q", data, at)
        at += 8
        if n > 16:
            continue                        # the text alone, in some other section
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, at)
            target = data[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx950" in target:
                yield data[m.start() + off:m.start() + off + size]


def _kernels(tmp_path):
    out = {}
    for k, obj in enumerate(_code_objects()):
        p = tmp_path / f"{k}.co"
        p.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(p)], check=True, capture_output=True, text=True).stdout
        for part in notes.split("- .agpr_count")[1:]:
            use = {key: int(x) for key, x in re.findall(r"\.(\w+):\s+(\d+)\n", part)}
            out[re.search(r"\.symbol:\s+(\S+)\.kd", part).group(1)] = use
    return out


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_state_copies_stay_in_registers(tmp_path):
    use, = [v for k, v in _kernels(tmp_path).items() if "k_copy_arrays" in k]
    assert use["group_segment_fixed_size"] == 0 and use["private_segment_fixed_size"] == 0
    assert use["vgpr_count"] >= 16
