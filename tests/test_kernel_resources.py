"""CPU: registers, scratch memory and LDS of the built library's kernels, from the notes of its
gfx950 code objects."""
import re
import struct
import subprocess

import pytest

from neuzip_amd import _build

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name -> fields of its metadata"""
    blob = open(_build.LIB_PATH, "rb").read()
    d = tmp_path_factory.mktemp("code")
    out = {}
    for k, m in enumerate(re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", blob)):
        at = m.start() + 32
        for _ in range(struct.unpack_from("<Q", blob, m.start() + 24)[0]):
            off, size, name = struct.unpack_from("<QQQ", blob, at)
            at += 24 + name
            if b"gfx950" not in blob[at - name:at]:
                continue
            path = d / f"{k}.co"
            path.write_bytes(blob[m.start() + off:m.start() + off + size])
            notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
            for part in notes.split("- .agpr_count:")[1:]:
                f = dict(re.findall(r"^\s+(\.\w+):\s+(\S+)", part, re.M))
                out[re.search(r"^\s+\.symbol:\s+(\S+)\.kd", part, re.M).group(1)] = f
    return out


def _of(kernels, stem, at_least):
    found = {k: f for k, f in kernels.items() if stem in k}
    assert len(found) >= at_least
    return found


def test_register_encode_kernels_do_not_spill(kernels):
    """The host sizes LDS by the wavefronts per SIMD unit that nz_enc_waves names; the registers
    (512 per lane and SIMD unit, given out by eights) have to allow them, without scratch memory."""
    found = _of(kernels, "nz_encode_kernel", 16)
    for name, f in found.items():
        groups = int(re.search(r"ELi(\d+)EE", name).group(1))
        waves = {8: 7, 16: 5, 32: 4, 36: 4}[groups]
        assert int(f[".vgpr_spill_count"]) == 0 and int(f[".private_segment_fixed_size"]) == 0, name
        assert 512 // (-(-int(f[".vgpr_count"]) // 8) * 8) >= waves, name


def test_kernels_that_decode_have_no_static_lds(kernels):
    """The one-read step takes the slot table, the start of the dynamic LDS, to be at LDS address 0."""
    found = _of(kernels, "nz_decode_", 136)
    for name, f in found.items():
        assert int(f[".group_segment_fixed_size"]) == 0, name
        assert int(f[".vgpr_spill_count"]) == 0 and int(f[".private_segment_fixed_size"]) == 0, name
