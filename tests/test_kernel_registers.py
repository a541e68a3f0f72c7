"""Registers of the kernels whose speed rests on how many of their wavefronts a SIMD holds, read from the metadata of the library's
own code objects (host only)."""
import re
import struct
import subprocess

import pytest

import floneum_amd as fa

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{symbol: {field: value}} of every kernel in the library."""
    data, found, at = open(fa.LIB_PATH, "rb").read(), {}, 0
    path = tmp_path_factory.mktemp("code") / "object"
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        (count,), pos = struct.unpack_from("<Q", data, at + 24), at + 32
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            name, pos = data[pos + 24:pos + 24 + length], pos + 24 + length
            if b"gfx950" in name:
                path.write_bytes(data[at + offset:at + offset + size])
                notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
                for entry in notes.split("  - .agpr_count:")[1:]:
                    fields = {k: int(v) for k, v in re.findall(r"\.([a-z_]+): +(\d+)\n", entry)}
                    found[re.search(r"\.name: +(\S+)\n", entry).group(1)] = dict(fields, agpr_count=int(entry.split()[0]))
        at += 1
    assert len(found) > 50
    return found


@pytest.mark.parametrize("kernel, wavefronts", [
    ("decode_mfma_f32_kernelILi96ELi1EE", 3), ("decode_mfma_f32_kernelILi128ELi1EE", 2), ("decode_mfma_f32_kernelILi64ELi1EE", 4),
    ("16rope_rows_kernel", 8), ("15row_jobs_kernel", 4),
])
def test_wavefronts_per_simd(kernels, kernel, wavefronts):
    """512 vector registers per SIMD lane, in steps of 8, and 800 scalar ones in steps of 16."""
    found = [v for k, v in kernels.items() if kernel in k]
    assert found
    for k in found:
        assert (k["vgpr_count"] + 7) // 8 * 8 * wavefronts <= 512, k
        assert (k["sgpr_count"] + 15) // 16 * 16 * wavefronts <= 800, k
        assert k["vgpr_spill_count"] == 0, k
