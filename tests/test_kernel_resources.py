"""Resources of the built kernels, from the metadata of libnbody_hip.so: kernels
whose values all fit the registers keep none of them in scratch memory."""
import os
import re
import struct
import subprocess

import pytest

from conftest import PKG

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def scratch(tmp_path_factory):
    """{kernel symbol: scratch bytes per work-item} of every gfx950 kernel."""
    with open(os.path.join(PKG, "libnbody_hip.so"), "rb") as f:
        lib = f.read()
    out, at = {}, lib.find(MAGIC)
    while at >= 0:
        (entries,) = struct.unpack_from("<Q", lib, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", lib, p)
            target = lib[p + 24:p + 24 + length].decode()
            p += 24 + length
            if "gfx950" not in target or size == 0:
                continue
            co = tmp_path_factory.mktemp("co") / "kernels.co"
            co.write_bytes(lib[at + offset:at + offset + size])
            notes = subprocess.run([READELF, "--notes", str(co)], capture_output=True, text=True,
                                   check=True).stdout
            for kernel in re.split(r"\n  - ", notes):
                private = re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel)
                symbol = re.search(r"\.symbol:\s+'?([\w$]+)\.kd", kernel)
                if private and symbol:
                    out[symbol.group(1)] = int(private.group(1))
        at = lib.find(MAGIC, at + 1)
    return out


@pytest.mark.parametrize("kernel,count", [("k_direct_f32c", 2), ("k_direct_f64f", 1),
                                          ("k_bh_exact_wave", 1)])
def test_no_scratch(scratch, kernel, count):
    sizes = {k: v for k, v in scratch.items() if kernel in k}
    assert len(sizes) == count, sizes
    assert set(sizes.values()) == {0}, sizes
