"""What the compiled kernels take, read from the gfx950 code objects inside the
built library: no codebook kernel keeps registers in scratch memory."""
import os
import re
import struct
import subprocess

import pytest

import rustyneedle_amd as rn

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data: bytes):
    """The gfx950 code objects of every offload bundle: after the magic a count,
    then per entry an offset from the bundle's start, a size and a named target."""
    at = data.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            target = data[entry + 24:entry + 24 + length]
            entry += 24 + length
            if target.endswith(b"gfx950") and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def scratch(tmp_path_factory):
    """Bytes of scratch a lane, by kernel."""
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    folder, found = tmp_path_factory.mktemp("objects"), {}
    with open(rn.LIB_PATH, "rb") as f:
        data = f.read()
    for i, blob in enumerate(_code_objects(data)):
        path = folder / f"{i}.co"
        path.write_bytes(blob)
        notes = subprocess.run([READELF, "--notes", str(path)], check=True, capture_output=True, text=True).stdout
        names = re.findall(r"^ +\.name: +(_Z\S+)", notes, re.M)
        sizes = re.findall(r"\.private_segment_fixed_size: +(\d+)", notes)
        assert len(names) == len(sizes)
        found.update(zip(names, map(int, sizes)))
    return found


def test_codebook_kernels_keep_no_registers_in_scratch(scratch):
    kernels = {n: b for n, b in scratch.items() if "cb_" in n}
    assert len(kernels) > 60
    assert not {n: b for n, b in kernels.items() if b}
