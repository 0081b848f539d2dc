"""CPU check of the scratch (private memory in HBM) and the registers of the built
kernels, read from the metadata of the library's own gfx950 code objects: a kernel
that the compiler gave room for its arguments in scratch, or many more registers
than it needs, runs slower, with the same results."""
import os
import re
import struct
import subprocess
import tempfile

import pytest

from amrclaw_amd import capi

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(blob):
    """The device code objects of the offload bundles in a shared library."""
    at = blob.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", blob, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, tlen = struct.unpack_from("<QQQ", blob, p)
            triple = blob[p + 24:p + 24 + tlen]
            p += 24 + tlen
            if b"gfx950" in triple and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, at + 1)


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
def test_scratch_of_the_kernels():
    scratch, vgprs = {}, {}
    blob = open(capi.LIBPATH, "rb").read()
    with tempfile.TemporaryDirectory() as d:
        for k, co in enumerate(code_objects(blob)):
            f = os.path.join(d, "%d.co" % k)
            open(f, "wb").write(co)
            notes = subprocess.run([READELF, "--notes", f], capture_output=True, text=True,
                                   check=True).stdout
            # (a kernel's keys stand in alphabetical order: its name before its
            # private_segment_fixed_size and vgpr_count)
            name = None
            for key, value in re.findall(r"\.(name|private_segment_fixed_size|vgpr_count):\s+(\S+)",
                                         notes):
                if key == "name":
                    name = value if value.startswith("_Z") else name
                elif name:
                    (vgprs if key == "vgpr_count" else scratch)[name] = int(value)
    fill = {n: v for n, v in scratch.items() if "fill_kernel" in n}
    assert len(fill) == 4 and len(scratch) > 100, (len(fill), len(scratch))
    # the kernels of every step; a few spilled scalar registers are no loss
    for part in ("fill_kernel", "update_kernel", "sweep3_tile", "pass3_", "xfer_kernel", "noalloc",
                 "finereg_kernel"):
        sizes = {n: v for n, v in scratch.items() if part in n}
        assert sizes and max(sizes.values()) <= 256, sizes
    assert max(fill.values()) <= 64, fill
    # four waves a SIMD: the fill waits for its loads
    assert max(vgprs[n] for n in fill) <= 128, {n: vgprs[n] for n in fill}
