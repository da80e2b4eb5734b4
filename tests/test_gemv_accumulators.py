"""CPU: the row accumulators of fused products.  A graph that captured a product writes to them
on every replay, so they outlive later calls that need more and a trim; and they are sized for the
next power of two of a call's activation rows, so that a product that has been made with five rows can be
captured with eight.  The library runs in a child process on the stand-in for the HIP runtime of
test_launch_forms.py, here with a switch for capture, the addresses that are given back, and the
kernel arguments of the last launch."""
import subprocess
import sys

import pytest

from test_launch_forms import CHILD, ROOT, RUNTIME

TRACKED = (RUNTIME
           .replace("int hipFree(void* p) { free(p); return 0; }",
                    "void* stub_freed[64]; int stub_nfreed;\n"
                    "int hipFree(void* p) { if (p) stub_freed[stub_nfreed++ & 63] = p; return 0; }")
           .replace("int* c) { *c = 0;", "int* c) { *c = stub_capturing;")
           .replace("int stub_cus, stub_n;", "int stub_cus, stub_n, stub_capturing; void* stub_acc;")
           # the first argument of a product is its batch: 24 bytes, then items whose fifth word is the accumulators
           .replace("{ stub_lds[stub_n++ & 63] = s;",
                    "{ stub_acc = ((void***)a)[0][3 + 4]; stub_lds[stub_n++ & 63] = s;"))

BODY = CHILD[:CHILD.index("got = {}")] + r"""
ctypes.c_int.in_dll(stub, "stub_capturing")  # all three are there: the stand-in is the tracked one
nfreed = ctypes.c_int.in_dll(stub, "stub_nfreed")
freed = (ctypes.c_void_p * 64).in_dll(stub, "stub_freed")
for chunks in (5000, 10000, 20000, 100000):  # two rows of 512 each
    store(h, b"w%d" % chunks, chunks)


def product(chunks, rows, capture=False):
    ctypes.c_int.in_dll(stub, "stub_capturing").value = capture
    rc = L.nz_manager_gemv_rows_batch(h, (ctypes.c_char_p * 1)(b"w%d" % chunks), 1, at, rows, 512, None,
                                      (ctypes.c_void_p * 1)(at), None)
    ctypes.c_int.in_dll(stub, "stub_capturing").value = 0
    assert rc == 0, m.last_error()
    return ctypes.c_void_p.in_dll(stub, "stub_acc").value


def given_back():
    return set(freed[: nfreed.value])
"""


@pytest.fixture(scope="module")
def child(tmp_path_factory):
    d = tmp_path_factory.mktemp("tracked")
    (d / "stub.c").write_text(TRACKED)
    subprocess.run(["gcc", "-shared", "-fPIC", "-w", "-o", str(d / "libstub.so"), str(d / "stub.c")], check=True)

    def run(code):
        res = subprocess.run([sys.executable, "-c", BODY + code, str(d / "libstub.so"), ROOT, "256"],
                             capture_output=True, text=True, timeout=120)
        assert res.returncode == 0, res.stderr

    return run


@pytest.mark.parametrize("captured_rows", [1, 3, 5, 8])
@pytest.mark.parametrize("then", ["product(10000, 8)", "product(20000, 8)", "product(20000, 1); product(100000, 2)",
                                  "L.nz_manager_trim(h)"])
def test_captured_accumulators_stay(child, captured_rows, then):
    child(f"""
product(10000, {captured_rows})
acc = product(10000, {captured_rows}, capture=True)
{then}
assert acc not in given_back()
if "trim" in {then!r}:
    assert product(10000, {captured_rows}) == acc  # and are still the ones in use
again = product(10000, {captured_rows}, capture=True)
L.nz_manager_destroy(h)
assert {{acc, again}} <= given_back()
""")


def test_capture_with_more_rows_than_the_calls_before(child):
    child("""
for chunks in (5000, 10000, 20000):  # 5 x 10000 rows fit the least that is allocated, 8 x 10000 do not
    for made, captured in ((3, (4, 2)), (5, (8, 6, 7, 1))):
        acc = product(chunks, made)
        for rows in captured:
            assert product(chunks, rows, capture=True) == acc
    for rows in (6, 8, 7, 5):
        assert product(chunks, rows) == acc
""")


def test_accumulators_no_graph_holds_are_given_back(child):
    child("""
first = product(10000, 8)
second = product(100000, 1)
assert first in given_back() and second not in given_back()
L.nz_manager_trim(h)
assert second in given_back()
""")
