"""What the built library says of itself without a GPU: the launch rules' choices (through
tests/cpp/launch_rules.cpp) and the kernels' resources, from the code objects' metadata."""
import os
import struct
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "tests", "cpp", "_build", "launch_rules")
LIB = os.path.join(ROOT, "umpalumpa_amd", "libumpalumpa_amd.so")

PAIR, CARRY, STAGED, CELLS = 1, 2, 3, 4


def ask(command, cases):
    """One answer (a list of words) per case (a dict of numbers)."""
    lines = [" ".join([command] + [f"{k}={v}" for k, v in c.items()]) for c in cases]
    r = subprocess.run([EXE], input="\n".join(lines) + "\n", capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr
    out = [line.split() for line in r.stdout.splitlines()]
    assert len(out) == len(lines)
    return out


def choices(cases):
    """(which kernel, workgroups, threads, dynamic LDS bytes, kernel symbol) per case."""
    return [(int(a), int(b), int(c), int(d), e) for a, b, c, d, e in ask("insert", cases)]


def kernel_metadata():
    """symbol -> metadata of every gfx950 kernel in the library (AMDGPU note of each code object)."""
    import msgpack
    data = open(LIB, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    out, at = {}, data.find(magic)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(magic))
        p = at + len(magic) + 8
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + n]
            p += 24 + n
            if b"gfx950" in name:
                out.update(_elf_kernels(data[at + offset:at + offset + size], msgpack))
        at = data.find(magic, at + 1)
    return out


def _elf_kernels(elf, msgpack):
    assert elf[:4] == b"\x7fELF"
    sections, = struct.unpack_from("<Q", elf, 0x28)
    entry, count = struct.unpack_from("<HH", elf, 0x3A)
    for k in range(count):
        h = sections + k * entry
        kind, = struct.unpack_from("<I", elf, h + 4)
        offset, = struct.unpack_from("<Q", elf, h + 0x18)
        if kind == 7:  # a note: name size, description size, type, name, description
            n, d, _ = struct.unpack_from("<III", elf, offset)
            start = offset + 12 + ((n + 3) & ~3)
            meta = msgpack.unpackb(elf[start:start + d], strict_map_key=False)
            return {m[".name"]: m for m in meta["amdhsa.kernels"]}
    return {}
