"""What the compiler made of kernels that fill a wave's registers, read from the built library's own notes: a spilled register is memory traffic that
the source does not show.  The column kernel in registers has every register of a lane in use at D = 256, and an epilogue that reads ahead tips it over."""
import os
import re
import struct
import subprocess

import pytest

from _mlstm_pkg import submodule

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


@pytest.fixture(scope="module")
def scratch(tmp_path_factory):
    """kernel -> bytes of scratch memory per lane"""
    image = open(submodule("_ffi").LIB_PATH, "rb").read()
    found = {}
    for n, bundle in enumerate(re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", image)):
        entry = bundle.end() + 8
        for _ in range(struct.unpack_from("<Q", image, bundle.end())[0]):
            at, size, name = struct.unpack_from("<QQQ", image, entry)
            entry += 24 + name
            if b"gfx950" in image[entry - name:entry]:
                out = tmp_path_factory.mktemp("code") / f"{n}.elf"
                out.write_bytes(image[bundle.start() + at:bundle.start() + at + size])
                notes = subprocess.run([READELF, "--notes", str(out)], capture_output=True, text=True, check=True).stdout
                found.update((k, int(b)) for k, b in re.findall(r"\.name: +(\w+)\n(?:.*\n)*? +\.private_segment_fixed_size: (\d+)", notes))
    return found


@pytest.mark.skipif(not os.path.exists(READELF), reason="no llvm-readelf")
@pytest.mark.parametrize("kernel,count", [
    ("cold_kernelIDF16bLi", 8),    # bf16, D = 128 and 256, split mode and not, dense and strided
    ("cold_kernelIDF16_Li128", 4),
    ("chunk_seq_kernel", 24),      # (launches of one with scratch memory go to other kernels)
])
def test_no_scratch_memory(scratch, kernel, count):
    sizes = {k: b for k, b in scratch.items() if kernel in k}
    assert len(sizes) == count and not any(sizes.values()), sizes
