"""The vector memory operations of a built kernel, by the windows between its barriers: what the scans'
hand-counted waits rest on.  Read from libcqgdn.so's gfx950 code with the ROCm disassembler."""

import re
import struct
import subprocess
from functools import lru_cache
from pathlib import Path

LIB = Path(__file__).resolve().parents[1] / "cq-pretrain_amd" / "cqgdn" / "libcqgdn.so"
OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects():
    """The gfx950 ELF images in the library's offload bundles."""
    data = LIB.read_bytes()
    for m in re.finditer(MAGIC, data):
        at = m.start()
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + n].decode()
            pos += 24 + n
            if "gfx950" in name and size:
                yield data[at + offset:at + offset + size]


@lru_cache(maxsize=None)
def instructions(symbol, directory):
    """The instructions (text) of the one kernel whose mangled name contains ``symbol``, in layout order."""
    for i, image in enumerate(_code_objects()):
        if symbol.encode() not in image:
            continue
        path = Path(directory) / f"image{i}.co"
        path.write_bytes(image)
        text = subprocess.run([str(OBJDUMP), "-d", str(path)], capture_output=True, text=True, check=True).stdout
        found = re.findall(r"^[0-9a-f]+ <(\S*%s\S*)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)" % re.escape(symbol), text,
                           re.M | re.S)
        assert len(found) == 1, [name for name, _ in found]
        return tuple(line.split("//")[0].strip() for line in found[0][1].splitlines() if line.strip())
    raise AssertionError(f"no kernel {symbol} in {LIB}")


def windows(symbol, directory):
    """Per window between barriers: a list of "copy" (global -> LDS), "load", "store", ("wait", n) and
    "read" (LDS), in layout order."""
    out = [[]]
    for ins in instructions(symbol, directory):
        op = ins.split()[0]
        if op == "s_barrier":
            out.append([])
        elif re.match(r"(buffer|global|flat)_load", op):
            out[-1].append("copy" if re.search(r"\blds\b", ins) else "load")
        elif re.match(r"(buffer|global|flat)_store", op):
            out[-1].append("store")
        elif re.match(r"(buffer|global|flat)_atomic", op):
            out[-1].append("atomic")
        elif op.startswith("ds_read"):
            out[-1].append("read")
        elif op == "s_waitcnt" and (m := re.search(r"vmcnt\((\d+)\)", ins)):
            out[-1].append(("wait", int(m[1])))
    return out
