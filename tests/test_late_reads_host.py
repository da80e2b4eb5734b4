"""CPU: what the host does for a read behind an in-place write that is still running.  On the write's own
stream it enqueues the read without waiting.  The library runs in a child process on the stand-in for
the HIP runtime of test_launch_forms.py, here with events that are not done until they are waited for."""
import subprocess
import sys

import pytest

from test_launch_forms import CHILD, ROOT, RUNTIME

RUNNING = (RUNTIME
           .replace("int hipEventQuery(void* e) { return 0; }", "int stub_done = 1; int hipEventQuery(void* e) { return stub_done ? 0 : 600; }")
           .replace("int hipEventSynchronize(void* e) { return 0; }",
                    "int stub_waits; int hipEventSynchronize(void* e) { ++stub_waits; stub_done = 1; return 0; }")
           .replace("int hipMalloc(void** p, size_t n) {", "int stub_allocs; int hipMalloc(void** p, size_t n) { ++stub_allocs;")
           .replace("int hipFree(void* p) {", "int hipFree(void* p) { ++stub_allocs;")
           + "int hipPeekAtLastError(void) { return 0; }\n"
             "int hipFuncSetAttribute(const void* f, int a, int v) { return 0; }\n")

BODY = CHILD[:CHILD.index("got = {}")] + r"""
done, waits, allocs = (ctypes.c_int.in_dll(stub, k) for k in ("stub_done", "stub_waits", "stub_allocs"))
PER_THREAD = 2  # hipStreamPerThread


def rewrite(name, n, stream):
    assert L.nz_manager_write_batch(h, (ctypes.c_char_p * 1)(name), (ctypes.c_void_p * 1)(at), (ctypes.c_uint64 * 1)(n), 1,
                                    m.DTYPE_BF16, stream) == 0, m.last_error()
    done.value = 0


def read(name, n, stream):
    # -> (did the host wait, did it allocate or free memory, launches)
    waits.value = allocs.value = launched.value = 0
    assert L.nz_manager_read(h, name, at, n, stream) == 0, m.last_error()
    return waits.value, allocs.value, launched.value


store(h, b"w", 40)
N = 40 * CHUNK
"""


@pytest.fixture(scope="module")
def child(tmp_path_factory):
    d = tmp_path_factory.mktemp("running")
    (d / "stub.c").write_text(RUNNING)
    subprocess.run(["gcc", "-shared", "-fPIC", "-w", "-o", str(d / "libstub.so"), str(d / "stub.c")], check=True)

    def run(code):
        res = subprocess.run([sys.executable, "-c", BODY + code, str(d / "libstub.so"), ROOT, "256"],
                             capture_output=True, text=True, timeout=120)
        assert res.returncode == 0, res.stderr

    return run


def test_a_read_waits_on_another_stream_and_on_a_handle_that_is_no_one_stream(child):
    child("""
rewrite(b"w", N, 64)
assert read(b"w", N, 64)[0] == 1  # the first time a read comes this soon it waits
for k in range(4):
    rewrite(b"w", N, 64)
    assert read(b"w", N, 64)[0] == 0
    assert read(b"w", N, 64)[0] == 0
    rewrite(b"w", N, 64)
    assert read(b"w", N, 128)[0] == 1
    assert read(b"w", N, 64)[0] == 0  # (known by now)
    rewrite(b"w", N, PER_THREAD)
    assert read(b"w", N, PER_THREAD)[0] == 1  # may be another thread's
""")


def test_reads_allocate_nothing(child):
    """The room that a read behind a write may need is the write's to find, and has a bound."""
    child("""
store(h, b"v", 80)
for name, n in ((b"w", N), (b"v", 2 * N), (b"w", N), (b"v", 2 * N)):
    for k in range(3):
        rewrite(name, n, 64)
        assert read(name, n, 64)[1] == 0
assert read(b"v", 2 * N, 64)[0] == 0 and read(b"w", N, 64)[1] == 0
# 135 million elements: more room than is kept for this, the read waits
big = 132000
store(h, b"b", big)
for k in range(3):
    rewrite(b"b", big * CHUNK, 64)
    assert read(b"b", big * CHUNK, 64)[:2] == (1, 0)
rewrite(b"w", N, 64)
assert read(b"w", N, 64)[:2] == (0, 0)
L.nz_manager_trim(h)  # gives the room back; the next write finds it again
rewrite(b"w", N, 64)
assert read(b"w", N, 64)[:2] == (0, 0)
L.nz_manager_destroy(h)
""")
