"""CPU: which ring a launch that decodes gets, and what LDS a fused product asks for.  Launches of at
most one workgroup per compute unit of the device in use decode with the one-read step and its wide
ring, 4 KiB per wavefront.  Larger ones have 2 KiB: dense output a ring of words (the two-read
step), fused products the narrow ring of prepared entries (the one-read step again); which of the
two is a matter of the kernel, not of its LDS.  Products of six to eight rows stage activations behind the
rings there, 2 KiB per row, where chunks have a segment for each row.  The library runs in a child
process on a stand-in for the HIP runtime (memory from the host, launches recorded and not run)."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r"""
#include <stdlib.h>
#include <string.h>
typedef struct { unsigned x, y, z; } dim3;
int stub_cus, stub_n;
unsigned long stub_lds[64];
static dim3 g_, b_;
static size_t s_;
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, void* st) { g_ = g; b_ = b; s_ = s; return 0; }
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, void** st) { *g = g_; *b = b_; *s = s_; *st = 0; return 0; }
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t s, void* st) { stub_lds[stub_n++ & 63] = s; return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int* v, int what, int d) { *v = stub_cus; return 0; }
int hipMalloc(void** p, size_t n) { *p = aligned_alloc(256, (n + 511) & ~(size_t)255); return !*p; }
int hipFree(void* p) { free(p); return 0; }
int hipHostMalloc(void** p, size_t n, unsigned f) { return hipMalloc(p, n); }
int hipHostFree(void* p) { free(p); return 0; }
int hipHostGetDevicePointer(void** d, void* h, unsigned f) { *d = h; return 0; }
int hipMemset(void* p, int v, size_t n) { memset(p, v, n); return 0; }
int hipMemsetAsync(void* p, int v, size_t n, void* st) { memset(p, v, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) { memcpy(d, s, n); return 0; }
int hipEventCreateWithFlags(void** e, unsigned f) { *e = (void*)1; return 0; }
int hipEventDestroy(void* e) { return 0; }
int hipEventQuery(void* e) { return 0; }
int hipEventRecord(void* e, void* st) { return 0; }
int hipEventSynchronize(void* e) { return 0; }
int hipStreamWaitEvent(void* st, void* e, unsigned f) { return 0; }
int hipStreamSynchronize(void* st) { return 0; }
int hipStreamIsCapturing(void* st, int* c) { *c = 0; return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipGetLastError(void) { return 0; }
"""

CHILD = r"""
import ctypes, importlib.util, json, os, struct, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # found before the real runtime
spec = importlib.util.spec_from_file_location("nz_lib", os.path.join(sys.argv[2], "neuzip_amd", "_lib.py"))
m = importlib.util.module_from_spec(spec)
spec.loader.exec_module(m)
L = m.load()
cus = int(sys.argv[3])
ctypes.c_int.in_dll(stub, "stub_cus").value = cus
launched = ctypes.c_int.in_dll(stub, "stub_n")
lds = (ctypes.c_ulong * 64).in_dll(stub, "stub_lds")
CHUNK, LANE = 1024, 16  # one wavefront per workgroup
buf = ctypes.create_string_buffer(1 << 16)
at = (ctypes.addressof(buf) + 255) & ~255  # stands for every device buffer: nothing is run


def form(call):
    launched.value = 0
    rc = call()
    assert rc == 0, m.last_error()
    return {32768 + 4096: "wide", 32768 + 2048: "2 KiB"}[lds[0]]


def store(mgr, name, chunks, segs=1):
    # a well-formed header and directory; the records stay empty
    rec = (64 + 4 * (chunks * segs + 1) + 15) & ~15
    total, chunk = rec + 16, CHUNK * segs
    comp = struct.pack("<6I4IQ4I", 0x315A4E41, 4, chunk * chunks, 0, chunk, LANE, chunks, chunks * segs, 64, rec, total,
                       0, 0, 0, 0)
    comp = ctypes.create_string_buffer(comp + bytes(total - 64), total)
    packed = ctypes.create_string_buffer(L.nz_packed_stored_bytes(chunk * chunks, 7, chunk, LANE))
    assert L.nz_manager_import(mgr, name, comp, total, packed, len(packed), None, 0, None) == 0, m.last_error()


h = ctypes.c_void_p()
assert L.nz_manager_create(0, 7, 0, CHUNK, LANE, ctypes.byref(h)) == 0
got = {}
for chunks in (cus, cus + 1):
    n = CHUNK * chunks
    name = b"w%d" % chunks
    store(h, name, chunks)
    names, ptrs, caps = (ctypes.c_char_p * 1)(name), (ctypes.c_void_p * 1)(at), (ctypes.c_uint64 * 1)(n)
    out = {
        "decode": lambda: L.nz_decode(at, 1 << 20, at, n, 7, CHUNK, LANE, at, at, 0, 0, None, None),
        "streaming decode": lambda: L.nz_decode(at, 1 << 20, at, n, 7, CHUNK, LANE, at, at, m.DECODE_STREAM_OUT, 0, None, None),
        "read": lambda: L.nz_manager_read(h, name, at, n, None),
        "read_batch": lambda: L.nz_manager_read_batch(h, names, ptrs, caps, 1, None),
        "product": lambda: L.nz_manager_gemv_batch(h, names, 1, at, 512, None, ptrs, None),
        "product of 8 rows": lambda: L.nz_manager_gemv_rows_batch(h, names, 1, at, 8, 512, None, ptrs, None),
        "gather": lambda: L.nz_manager_gather_rows(h, name, at, chunks, CHUNK, at, None),
    }
    got["at the line" if chunks == cus else "above"] = {k: form(f) for k, f in out.items()}
    for segs in (4, 6, 8):
        store(h, b"s%d" % segs, chunks, segs)
        for rows in range(1, 9):
            launched.value = 0
            assert L.nz_manager_gemv_rows_batch(h, (ctypes.c_char_p * 1)(b"s%d" % segs), 1, at, rows, 512, None, ptrs, None) == 0
            got["%d segments, %d rows, %s" % (segs, rows, "line" if chunks == cus else "above")] = lds[0]
print(json.dumps(got))
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    d = tmp_path_factory.mktemp("stub")
    (d / "stub.c").write_text(RUNTIME)
    subprocess.run(["gcc", "-shared", "-fPIC", "-w", "-o", str(d / "libstub.so"), str(d / "stub.c")], check=True)
    return str(d / "libstub.so")


@pytest.mark.parametrize("cus", [256, 32])  # the whole device, one of eight partitions
def test_wide_ring_up_to_one_workgroup_per_compute_unit(runtime, cus):
    res = subprocess.run([sys.executable, "-c", CHILD, runtime, ROOT, str(cus)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stderr
    got = json.loads(res.stdout)
    line, above = got.pop("at the line"), got.pop("above")
    assert line.pop("streaming decode") == "2 KiB"
    assert set(line.values()) == {"wide"} and set(above.values()) == {"2 KiB"}, (line, above)
    for segs in (4, 6, 8):
        for rows in range(1, 9):
            staged = 2048 * rows if rows >= 6 and segs >= rows else 0
            assert got.pop(f"{segs} segments, {rows} rows, line") == 32768 + 4096 * segs
            assert got.pop(f"{segs} segments, {rows} rows, above") == 32768 + 2048 * segs + staged
    assert not got
