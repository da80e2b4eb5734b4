"""CPU: into how many workgroups a chunk is shared out, and the rings these ask for: the largest power of
two of workgroups per chunk that the compute units have room for, up to one per segment.  (The stand-in for the
HIP runtime of test_launch_forms.py, which here records grids as well.)"""
import json
import subprocess
import sys

import pytest

from test_launch_forms import CHILD, ROOT, RUNTIME

GRIDS = (RUNTIME.replace("unsigned long stub_lds[64];", "unsigned long stub_lds[64]; unsigned stub_grid[64];")
         .replace("{ stub_lds[stub_n++ & 63] = s;", "{ stub_grid[stub_n & 63] = g.x; stub_lds[stub_n++ & 63] = s;"))

BODY = CHILD[:CHILD.index("got = {}")] + r"""
grids = (ctypes.c_uint * 64).in_dll(stub, "stub_grid")
got = []
for segs in range(1, 9):
    for chunks in (1, cus // 8, cus // 8 + 1, cus // 4, cus // 4 + 1, cus // 2, cus // 2 + 1, cus):
        name = b"p%d_%d" % (segs, chunks)
        store(h, name, chunks, segs)
        n = CHUNK * segs * chunks
        names, ptrs, caps = (ctypes.c_char_p * 1)(name), (ctypes.c_void_p * 1)(at), (ctypes.c_uint64 * 1)(n)
        out = []
        for call in (lambda: L.nz_manager_read(h, name, at, n, None),
                     lambda: L.nz_manager_read_batch(h, names, ptrs, caps, 1, None),
                     lambda: L.nz_manager_gemv_batch(h, names, 1, at, 512, None, ptrs, None),
                     lambda: L.nz_manager_gemv_rows_batch(h, names, 1, at, 8, 512, None, ptrs, None)):
            launched.value = 0
            assert call() == 0, m.last_error()
            out.append([grids[0], lds[0]])
        launched.value = 0
        assert L.nz_decode(at, 1 << 20, at, n, 7, CHUNK * segs, LANE, at, at, m.DECODE_STREAM_OUT, 0, None, None) == 0
        got.append([segs, chunks, out, grids[0]])
print(json.dumps(got))
"""


@pytest.mark.parametrize("cus", [256, 32])
def test_chunks_are_shared_out_where_compute_units_are_left(tmp_path, cus):
    (tmp_path / "stub.c").write_text(GRIDS)
    subprocess.run(["gcc", "-shared", "-fPIC", "-w", "-o", str(tmp_path / "libstub.so"), str(tmp_path / "stub.c")], check=True)
    res = subprocess.run([sys.executable, "-c", BODY, str(tmp_path / "libstub.so"), ROOT, str(cus)],
                         capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stderr
    for segs, chunks, launches, streaming in json.loads(res.stdout):
        parts = max(p for p in (1, 2, 4, 8) if p <= segs and (p == 1 or p * chunks <= cus))
        rings = segs if parts == 1 else -(-segs // parts) + 1
        for grid, lds in launches:
            assert (grid, lds) == (parts * chunks, 32768 + 4096 * rings), (segs, chunks)
        assert streaming == chunks  # streaming stores: memory-bound, one workgroup per chunk
