"""Runs a snippet against libplk.so with hip_record.cpp in the place of the HIP runtime, in a
process of its own (CPU only)."""
import functools
import json
import os
import struct
import subprocess
import sys
import tempfile
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
READELF = "/opt/rocm/llvm/bin/llvm-readelf"

PRELUDE = """
import ctypes, json, sys
sys.path[:0] = [{root!r}, {tests!r}]
rec = ctypes.CDLL({stub!r}, mode=ctypes.RTLD_GLOBAL)
for name in ("rec_lds", "rec_blocks", "rec_threads", "rec_bytes"):
    getattr(rec, name).restype = ctypes.c_long
rec.rec_name.restype = ctypes.c_char_p
import numpy as np
import gems_amd as G
import support as S

def launches():
    out = [(rec.rec_name(i).decode(), rec.rec_lds(i), rec.rec_blocks(i)) for i in range(rec.rec_count())]
    rec.rec_clear()
    return out

def called(f, *a, **k):
    try:
        f(*a, **k)
        return 0
    except G.PlkError as e:
        return e.code
"""


KEEP = tempfile.TemporaryDirectory()  # until the tests end


@functools.lru_cache(maxsize=None)
def stub():
    out = os.path.join(KEEP.name, "hip_record.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "gems_amd", "csrc"),
                    os.path.join(ROOT, "tests", "hip_record.cpp"), "-o", out], check=True, timeout=300)
    return out


def run(code):
    """The JSON that the snippet prints in its last line."""
    text = PRELUDE.format(root=ROOT, tests=os.path.join(ROOT, "tests"), stub=stub()) + textwrap.dedent(code)
    r = subprocess.run([sys.executable, "-c", text], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout.strip().split("\n")[-1])


@functools.lru_cache(maxsize=None)
def kernel_notes():
    """Kernel name -> (bytes of its own LDS arrays, vector registers), from the notes of the device
    code built here."""
    with open(os.path.join(ROOT, "gems_amd", "libplk.so"), "rb") as f:
        data = f.read()
    magic, found, at = b"__CLANG_OFFLOAD_BUNDLE__", {}, -1
    while (at := data.find(magic, at + 1)) >= 0:
        pos = at + len(magic) + 8
        for _ in range(struct.unpack_from("<Q", data, at + len(magic))[0]):
            off, size, length = struct.unpack_from("<QQQ", data, pos)
            if b"gfx950" in data[pos + 24:pos + 24 + length]:
                with tempfile.NamedTemporaryFile() as elf:
                    elf.write(data[at + off:at + off + size])
                    elf.flush()
                    notes = subprocess.run([READELF, "--notes", elf.name], check=True, capture_output=True, text=True).stdout
                kernel = {}
                for line in notes.split("\n"):
                    if line.startswith("  - "):
                        kernel = {}
                    if line.startswith(("    .", "  - .")):
                        key, _, value = line[4:].partition(":")
                        kernel[key] = value.strip()
                    if line.startswith("    .wavefront_size:"):
                        found[kernel[".name"]] = int(kernel[".group_segment_fixed_size"]), int(kernel[".vgpr_count"])
            pos += 24 + length
    return found


def static_lds():
    return {name: lds for name, (lds, _) in kernel_notes().items()}
