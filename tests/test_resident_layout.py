"""The one-launch time loop as built (no GPU needed): where its LDS arrays begin."""
import os
import re
import struct
import subprocess

from ifos_amd import build as B

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def kernel_metadata(tmp_path):
    """(name, static LDS bytes) of every kernel in the library's gfx950 code objects."""
    blob = open(B.LIB, "rb").read()
    magic, found, pos = b"__CLANG_OFFLOAD_BUNDLE__", [], 0
    while (pos := blob.find(magic, pos)) >= 0:
        count, = struct.unpack_from("<Q", blob, pos + len(magic))
        at = pos + len(magic) + 8
        for _ in range(count):
            offset, size, chars = struct.unpack_from("<QQQ", blob, at)
            triple = blob[at + 24:at + 24 + chars]
            at += 24 + chars
            if not triple.endswith(b"gfx950") or not size:
                continue
            obj = tmp_path / "code.o"
            obj.write_bytes(blob[pos + offset:pos + offset + size])
            notes = subprocess.run([READELF, "--notes", str(obj)], check=True, stdout=subprocess.PIPE, text=True).stdout
            found += [(m[2], int(m[1])) for m in
                      re.finditer(r"\.group_segment_fixed_size: *(\d+).*?\.name: *(\S+)", notes, re.S)]
        pos += len(magic)
    return found


def test_lds_arrays_begin_aligned(tmp_path):
    """The dynamic LDS array of a workgroup begins where the static part ends,
    and the FP64 reciprocals of the absorbing profiles sit in it at even float
    indices: its base has to be a multiple of 8 bytes."""
    sizes = [size for name, size in kernel_metadata(tmp_path) if "k_resident" in name]
    assert len(sizes) > 60  # stencil orders x mechanisms x rows per thread
    assert all(size % 8 == 0 for size in sizes), sorted(set(sizes))


def test_material_loads_stay_in_the_grid(tmp_path):
    """Rows of cells past the grid's last row, which the lowest tiles hold, read
    the materials of a cell that exists."""
    exe = tmp_path / "bounds"
    lib = os.path.dirname(B.LIB)
    subprocess.run([B.HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-I" + B.CSRC,
                    "-I" + os.path.join(B.ROOT, "include"), "-x", "hip",
                    os.path.join(B.ROOT, "tests", "c", "resident_bounds.cpp"), "-o", str(exe), "-L" + lib,
                    "-lifos2d_hip", "-Wl,-rpath," + lib], check=True)
    plans, outside, unguarded = map(int, subprocess.run([str(exe)], check=True, stdout=subprocess.PIPE,
                                                        text=True).stdout.split())
    assert plans > 200 and unguarded > 0  # some rows do lie past the padding
    assert outside == 0
