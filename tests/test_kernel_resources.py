"""What the compiler made of the kernels, read from the metadata of the built library."""
import os
import re
import subprocess

import pytest

from hetuctr_amd import build

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 code objects of a shared library: every bundle lists (offset, size, target) of its parts."""
    data, at = open(path, "rb").read(), 0
    number = lambda p: int.from_bytes(data[p:p + 8], "little")
    while (at := data.find(MAGIC, at)) >= 0:
        entry = at + len(MAGIC) + 8
        for _ in range(number(at + len(MAGIC))):
            offset, size, length = number(entry), number(entry + 8), number(entry + 16)
            target = data[entry + 24:entry + 24 + length]
            entry += 24 + length
            if size and target.endswith(b"gfx950"):
                yield data[at + offset:at + offset + size]
        at += len(MAGIC)


@pytest.mark.skipif(not os.path.exists(READELF) or not os.path.exists(build.LIB), reason="needs the built library and llvm-readelf")
def test_no_kernel_uses_scratch_memory(tmp_path):
    # Scratch means registers spilled, or kernel arguments copied because something indexed or passed them in a way the
    # compiler could not follow: a spill of one register made the push of a 53 k-key batch 20.2 -> 22.3 us, records copied
    # to scratch a push of 306 us 4150.
    kernels = {}
    for i, obj in enumerate(code_objects(build.LIB)):
        f = tmp_path / ("%d.o" % i)
        f.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(f)], stdout=subprocess.PIPE, text=True, check=True).stdout
        names = re.findall(r"^\s+\.symbol:\s+'?(\S+?)\.kd'?$", notes, re.M)
        sizes = re.findall(r"^\s+\.private_segment_fixed_size:\s+(\d+)$", notes, re.M)
        assert len(names) == len(sizes)
        kernels.update(zip(names, map(int, sizes)))
    assert len(kernels) > 400
    assert not {n: s for n, s in kernels.items() if s}
