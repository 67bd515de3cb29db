"""The products whose activation tiles go straight into LDS publish a tile with a counted wait in front of a barrier.  The count holds only if the compiled step has the
loads that it counts on, so the compiled steps are counted: in the code objects of the built library, on the host."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "xfastertransformer_amd", "libxft_hip.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    with open(path, "rb") as f:
        data = f.read()
    at = data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(n):
            offset, size, name = struct.unpack_from("<QQQ", data, entry)
            if data[entry + 24:entry + 24 + name].endswith(b"gfx950"):
                yield data[at + offset:at + offset + size]
            entry += 24 + name
        at = data.find(MAGIC, at + 1)


def steps(listing):
    """(kernel, requests into LDS, accesses behind the last of them, all accesses, what the wait leaves) of every barrier behind requests"""
    kernel, waits = None, None
    requests = behind = accesses = 0
    for line in listing:
        head = re.match(r"<(\S+)>:", line)
        if head:
            kernel = head.group(1) if "qgemm_direct_kernel" in head.group(1) else None
        op = line.strip()
        if kernel is None:
            continue
        if head or op.startswith(("s_branch", "s_endpgm")):
            requests = behind = accesses = 0
        elif op.startswith("global_load_lds"):
            requests, behind, accesses = requests + 1, 0, accesses + 1
        elif re.match(r"(global|buffer|flat|scratch)_(load|store)", op):
            behind, accesses = behind + 1, accesses + 1
        elif op.startswith("s_waitcnt"):
            left = re.search(r"vmcnt\((\d+)\)", op)
            waits = int(left.group(1)) if left else waits
        elif op.startswith("s_barrier"):
            if requests:
                yield kernel, requests, behind, accesses, waits
            requests = behind = accesses = 0


def too_lax(kernel, requests, behind, accesses, left):
    """Four-bit kinds (two tiles in LDS) publish the step's own tile, the others that of the step before."""
    kind = int(re.search(r"qgemm_direct_kernelILi(\d)E", kernel).group(1))
    return left > (behind if kind in (1, 2) else accesses)


def test_counted_waits_cover_what_they_publish(tmp_path):
    objdump = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin:" + os.environ.get("PATH", ""))
    if not objdump or not os.path.exists(LIB):
        pytest.skip("needs the built library and llvm-objdump")
    found = []
    for i, blob in enumerate(code_objects(LIB)):
        if b"qgemm_direct_kernel" not in blob:
            continue
        path = tmp_path / f"{i}.co"
        path.write_bytes(blob)
        names = set(re.findall(rb"_ZN6xfthip\w*qgemm_direct_kernel\w+Eii(?!\w)", blob))
        listing = subprocess.run([objdump, "-d", "--no-show-raw-insn", "--no-leading-addr", "--disassemble-symbols=" + ",".join(sorted(n.decode() for n in names)), str(path)],
                                 capture_output=True, text=True, check=True).stdout.splitlines()
        found += list(steps(listing))
    kinds = {re.search(r"ILi(\d)E", s[0]).group(1) for s in found}
    assert len(kinds) >= 4 and len({s[0] for s in found}) >= 30
    assert not [s for s in found if too_lax(*s)]
