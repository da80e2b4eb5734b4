"""CPU: the walk over the full groups of a segment waits for memory at the end of a group, not among its steps.
Packed bytes and normalizer bytes are loaded two groups ahead of their use; a wait in front of the steps is
for a load that has just been issued, or for a path that has nothing to do with this one, and costs up to a tenth
of a read.  From the code of the built library's gfx950 kernels."""
import re
import struct
import subprocess

import pytest

from neuzip_amd import _build

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    """name -> instructions of every kernel with dense output"""
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
            if b"nz_decode_kernel" not in path.read_bytes():
                continue
            text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], capture_output=True, text=True, check=True).stdout
            for part in re.split(r"(?m)^[0-9a-f]+ <", text)[1:]:
                name = part[:part.index(">")]
                if "nz_decode_kernel" in name or "nz_decode_batch_kernel" in name:
                    out[name] = [line.split("//")[0].strip() for line in part.split("\n")[1:]]
    return out


def _groups(instructions):
    """for every 16-byte store: what is between it and the branch or the refill of the ring before it, as LDS reads and
    waits for memory"""
    window = []
    for x in instructions:
        if x.startswith(("s_cbranch", "s_branch", "ds_write")):
            window = []
        elif x.startswith("ds_read"):
            window.append("read")
        elif x.startswith("s_waitcnt") and "vmcnt" in x:
            window.append("wait")
        elif x.startswith("global_store_dwordx4"):
            yield window
            window = []


def test_no_wait_for_memory_among_the_steps_of_a_group(code):
    assert len(code) == 4 * 2 * 6  # precisions, one tensor and several, forms
    for name, instructions in code.items():
        early = []
        for window in _groups(instructions):
            # (four reads or more: the end of a decoded group)
            if window.count("read") >= 4 and "wait" in window and window[window.index("wait"):].count("read") > 2:
                early.append(window)
        # with normalizers one: the odd last group of a segment with groups of fewer than eight elements, once
        norm = re.search(r"ILi\dELb(\d)E", name).group(1) == "1"
        assert len(early) <= norm, (name, early)
