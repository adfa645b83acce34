"""Register budgets of the built kernels: those whose inner loops keep a net's
activations in registers must not spill them to scratch memory (each tile would
move them through the caches again).  Read from the kernel descriptors' notes in
the built library; no GPU."""

import os
import re
import shutil
import struct
import subprocess

import pytest

from deepmd_amd import build

READELF = next((p for p in (os.path.join(build.ROCM, "llvm", "bin", "llvm-readelf"),
                            shutil.which("llvm-readelf") or "") if os.path.exists(p)), None)
pytestmark = pytest.mark.skipif(READELF is None or not os.path.exists(build.LIB),
                                reason="no llvm-readelf or no built library")


@pytest.fixture(scope="module")
def scratch(tmp_path_factory):
    """{mangled kernel name: bytes of scratch a lane}"""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    data = open(build.LIB, "rb").read()
    tmp = tmp_path_factory.mktemp("co")
    out = {}
    for k, m in enumerate(re.finditer(re.escape(magic), data)):
        pos = m.start() + len(magic)
        n, = struct.unpack_from("<Q", data, pos)
        pos += 8
        if n > 8:
            continue
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, pos)
            ident = data[pos + 24:pos + 24 + idlen]
            pos += 24 + idlen
            if b"gfx950" not in ident or size == 0:
                continue
            path = tmp / f"{k}.co"
            path.write_bytes(data[m.start() + off:m.start() + off + size])
            text = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True,
                                  check=True).stdout
            for blk in re.split(r"\n\s+- \.a", text):
                name = re.search(r"\.name:\s+'?(_Z\S+k_\w+?\S*?)'?\n", blk)
                priv = re.search(r"\.private_segment_fixed_size:\s+(\d+)", blk)
                if name and priv:
                    out[name.group(1)] = int(priv.group(1))
    assert out, "no kernels found in the library"
    return out


@pytest.mark.parametrize("kernel,limit", [
    # FP64 embedding: a few values around the call of an activation other than
    # tanh (96 bytes); spilled activations were 900 to 1,500
    ("k_fwd64", 128), ("k_bwd64", 128),
    # split FP16, nets in LDS or from memory: a few values outside the tile loop
    ("k_fwd2", 96), ("k_bwd2", 96),
])
def test_scratch(scratch, kernel, limit):
    mine = {n: b for n, b in scratch.items() if kernel in n}
    assert mine, kernel
    assert max(mine.values()) <= limit, sorted(mine.items(), key=lambda x: -x[1])[:3]
