"""What the compiler made of the kernels, read from the metadata of the built library."""
import os
import re
import subprocess

import pytest

from hetuctr_amd import build

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
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


def kernel_code(listing):
    """(name, first address, [(address, instruction, operands, what follows the address)]) of every function of a listing."""
    name, start, body = None, 0, []
    for line in listing.splitlines():
        if m := re.match(r"^([0-9a-f]+) <(\S+)>:", line):
            if name:
                yield name, start, body
            name, start, body = m.group(2), int(m.group(1), 16), []
        elif name and (m := re.match(r"^\s+(\S+)\s*(.*?)\s*//\s*([0-9A-F]+):(.*)$", line)):
            body.append((int(m.group(3), 16), m.group(1), m.group(2), m.group(4)))
    if name:
        yield name, start, body


def early_barriers(start, body):
    """Addresses of the barriers that some path reaches with LDS operations of the wave still under way."""
    at = {address: i for i, (address, *_) in enumerate(body)}
    after = [[] for _ in body]
    for i, (_, op, _, rest) in enumerate(body):
        if op.startswith("s_endpgm"):
            continue
        if op.startswith(("s_branch", "s_cbranch")):
            offset = re.search(r"<[^>+]+(?:\+0x([0-9a-f]+))?>", rest).group(1)
            after[i].append(at[start + int(offset or "0", 16)])
        if not op.startswith("s_branch") and i + 1 < len(body):
            after[i].append(i + 1)
    under_way, todo = [False] * len(body), list(range(len(body)))
    while todo:
        i = todo.pop()
        _, op, operands, _ = body[i]
        if op.startswith("ds_") and not op.startswith(("ds_bpermute", "ds_permute", "ds_swizzle", "ds_nop")):
            left = True
        elif op == "s_waitcnt" and (operands.strip() == "0" or "lgkmcnt(0)" in operands):
            left = False
        else:
            left = under_way[i]
        for k in after[i]:
            if left and not under_way[k]:
                under_way[k] = True
                todo.append(k)
    return [hex(body[i][0]) for i in range(len(body)) if body[i][1].startswith("s_barrier") and under_way[i]]


@pytest.mark.skipif(not os.path.exists(OBJDUMP) or not os.path.exists(build.LIB), reason="needs the built library and llvm-objdump")
def test_every_barrier_waits_for_the_lds(tmp_path):
    # The compiler may drop the wait in front of a barrier that opens a loop, and a wave then passes it before what it wrote is
    # in LDS: the sums of long runs lost a chunk of rows once in some thousand steps that way.
    early, barriers = {}, 0
    for i, obj in enumerate(code_objects(build.LIB)):
        f = tmp_path / ("%d.o" % i)
        f.write_bytes(obj)
        listing = subprocess.run([OBJDUMP, "-d", str(f)], stdout=subprocess.PIPE, text=True, check=True).stdout
        for name, start, body in kernel_code(listing):
            barriers += sum(op.startswith("s_barrier") for _, op, _, _ in body)
            if found := early_barriers(start, body):
                early[name] = found
    assert barriers > 1000
    assert not early
