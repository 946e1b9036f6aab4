"""What the compiler recorded of the built kernels (the code objects' metadata): none spills a vector register or has
scratch memory.  A reload from scratch waits for every DMA in flight, in the GEMMs' k-loops above all."""
import os
import re
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "umdk_amd", "lib", "libcamhip.so")
READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(blob):
    """The gfx950 code objects of the library's offload bundles: magic, u64 count, then per entry u64 offset (from the
    magic), u64 size, u64 length of its target's name, the name."""
    at = blob.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", blob, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", blob, p)
            if b"gfx950" in blob[p + 24:p + 24 + ln]:
                yield blob[at + off:at + off + size]
            p += 24 + ln
        at = blob.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    from umdk_amd import _lib
    _lib.lib()  # (its missing-library message first)
    d, found = tmp_path_factory.mktemp("co"), {}
    for i, co in enumerate(code_objects(open(LIB, "rb").read())):
        f = d / f"{i}.co"
        f.write_bytes(co)
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
        for k in re.split(r"\n  - \.a", notes)[1:]:
            get = lambda key: re.search(rf"\n\s+\.{key}:\s+(\S+)", k).group(1)  # noqa: E731
            found[get("name")] = (int(get("vgpr_spill_count")), int(get("private_segment_fixed_size")))
    return found


def test_no_kernel_spills_vector_registers(kernels):
    assert sum("gmm" in k for k in kernels) >= 16
    assert {k: v for k, v in kernels.items() if v != (0, 0)} == {}
