"""Registers and scratch of the built kernels, read from the metadata of the library's own code objects:
the tiles whose launch rules count on two resident blocks a CU must fit that often, without spills."""
import os
import re
import shutil
import struct
import subprocess

import pytest

import splathip

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(path):
    """The gfx950 ELF images of every offload bundle in the library."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        p = at + len(MAGIC)
        (n,) = struct.unpack_from("<Q", data, p)
        p += 8
        if n < 16:
            for _ in range(n):
                off, size, tl = struct.unpack_from("<QQQ", data, p)
                triple = data[p + 24:p + 24 + tl].decode()
                p += 24 + tl
                if "gfx950" in triple and size:
                    yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Kernel name -> (registers, bytes of scratch)."""
    if not os.path.exists(splathip.LIB_PATH) or not os.path.exists(READELF):
        pytest.skip("no built library or no llvm-readelf")
    out = {}
    tmp = tmp_path_factory.mktemp("objects")
    for k, image in enumerate(_code_objects(splathip.LIB_PATH)):
        path = tmp / f"{k}.elf"
        path.write_bytes(image)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for block in re.split(r"\n\s*- \.agpr_count", notes)[1:]:
            get = lambda key: re.search(rf"\.{key}:\s*(\S+)", block).group(1)
            out[get("name")] = (int(get("vgpr_count")), int(get("private_segment_fixed_size")))
    assert out
    return out


def test_fp32_128x128_tiles_fit_twice_a_cu(kernels):
    """512 registers a SIMD lane: two blocks of four waves a CU take at most 256 each."""
    tiles = {k: v for k, v in kernels.items() if "gemm_mfma_kernelIfLi128ELi128E" in k}
    assert len(tiles) >= 8
    for name, (registers, scratch) in tiles.items():
        assert registers <= 256 and scratch == 0, (name, registers, scratch)


def test_fp32_attention_fits_twice_a_cu(kernels):
    found = {k: v for k, v in kernels.items() if "attn_f32_kernel" in k}
    assert len(found) == 2
    for name, (registers, scratch) in found.items():
        assert registers <= 256 and scratch == 0, (name, registers, scratch)


def test_no_fp32_gemm_tile_spills(kernels):
    """A spilled register is re-read in the k-loop and waits for every load in flight."""
    tiles = {k: v for k, v in kernels.items() if "gemm_mfma_kernelIf" in k}
    assert len(tiles) >= 32
    assert not {k: v for k, v in tiles.items() if v[1] != 0}
