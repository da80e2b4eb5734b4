"""Fused products of matrices whose rows are not whole groups of 512 elements: rows that end inside a
group, inside one segment or shared by several, a last group that the tensor does not fill."""
import ctypes

import numpy as np
import pytest

from conftest import bf16_bits_normal, closed_form_recon

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _weight(rows, cols, kind, seed):
    if kind == "raw":  # exponents that do not compress, none of them 255
        rng = np.random.default_rng(seed)
        e = rng.integers(100, 140, rows * cols) if seed & 1 else rng.integers(1, 250, rows * cols)
        bits = (e << 7 | rng.integers(0, 128, rows * cols) | rng.integers(0, 2, rows * cols) << 15).astype(np.uint16)
    else:
        bits = bf16_bits_normal(rows * cols, seed)
    return torch.from_numpy(bits.view(np.int16).copy()).cuda().view(torch.bfloat16).view(rows, cols), bits


def _product(mgr, h, x, out_features, bias=None):
    be = mgr._be
    rows = x.numel() // x.shape[-1]
    y = torch.full((rows * out_features + 8,), 7.0, dtype=torch.bfloat16, device="cuda")
    be._product(be._L.nz_manager_linear_rows_batch, (ctypes.c_char_p * 1)(h.encode()), x, [bias], [y], rows)
    assert bool((y[rows * out_features:] == 7.0).all())
    return y[:rows * out_features].view(rows, out_features)


def _check(y, bits, x, bias, s):
    """bf16 results of fp32 partial sums: half a unit in the last place of the result (2^-9 of it, doubled) and
    2^-24 per addition of the magnitudes' sum, of which a lane makes at most a few hundred."""
    w = (closed_form_recon(bits, s).astype(np.uint32) << 16).view(np.float32).astype(np.float64).reshape(y.shape[1], -1)
    xv = x.double().cpu().numpy().reshape(y.shape[0], -1)
    ref = xv @ w.T + (0 if bias is None else bias.double().cpu().numpy())
    tol = 2.0 ** -8 * np.abs(ref) + 1e-5 * (np.abs(xv) @ np.abs(w).T)
    err = np.abs(y.double().cpu().numpy() - ref)
    assert np.all(err <= tol), float(np.max(err / tol))


@pytest.mark.parametrize("s", [7, 3, 1, 0])
@pytest.mark.parametrize("rows,cols,kind,chunk,lane", [
    (1, 520, "normal", 0, 0),           # one row, a group and a lane
    (37, 520, "normal", 0, 0),          # a boundary in almost every group
    (300, 1016, "normal", 0, 0),        # a lane short of two groups
    (129, 1032, "raw", 0, 0),
    (64, 4104, "normal", 0, 0),
    (1000, 1160, "normal", 32768, 64),  # rows begin in the middle of short segments
    (50, 16392, "normal", 0, 0),        # rows longer than a segment
    (9, 40008, "normal", 0, 0),         # ... than two
    (70, 5000, "raw", 8192, 16),        # ... and of five short segments
    (257, 512, "normal", 0, 0),         # whole groups all the same
])
def test_products_of_any_row_length(rows, cols, kind, chunk, lane, s):
    import neuzip_amd

    mgr = neuzip_amd.Manager(precision=s, chunk_size=chunk or None, lane_symbols=lane)
    w, bits = _weight(rows, cols, kind, rows + s)
    h = mgr.write(w)
    g = torch.Generator(device="cuda").manual_seed(cols)
    x = torch.randn(8, cols, device="cuda", generator=g).to(torch.bfloat16)
    if kind == "raw":
        x *= 2.0 ** -100 if (rows + s) % 2 == 0 else 1.0  # keep the sums finite
    bias = torch.randn(rows, device="cuda", generator=g).to(torch.bfloat16)
    print(f"case {rows}x{cols} {kind} {chunk}/{lane} s={s}", flush=True)
    one = [_product(mgr, h, x[m].contiguous(), rows) for m in range(8)]
    for m in (0, 7):
        _check(one[m], bits, x[m], None, s)
    _check(_product(mgr, h, x[0].contiguous(), rows, bias), bits, x[0], bias, s)
    for m_rows in (2, 5, 8):
        y = _product(mgr, h, x[:m_rows].contiguous(), rows)
        for m in range(m_rows):
            assert torch.equal(y[m].view(torch.int16), one[m][0].view(torch.int16)), (m_rows, m)
    mgr._be.check()


@pytest.mark.parametrize("norm", [1, 8, 512])
def test_products_of_any_row_length_with_normalizers(norm):
    import neuzip_amd

    mgr = neuzip_amd.Manager(precision=3, normalizer_size=norm)
    rows, cols = 200, 1160
    h = mgr.write(_weight(rows, cols, "normal", norm)[0])
    x = torch.randn(cols, device="cuda").to(torch.bfloat16)
    y = _product(mgr, h, x, rows)[0].double()
    w = mgr.read(h).double()
    ref = w @ x.double()
    assert bool(((y - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5 * (w.abs() @ x.double().abs())).all())
    mgr._be.check()


def test_a_row_does_not_leak_into_its_neighbours():
    import neuzip_amd

    rows, cols = 96, 1000
    w = torch.randn(rows, cols, device="cuda").to(torch.bfloat16)
    for k in (5, 40, rows - 1):
        w[k] = float("inf")
    mgr = neuzip_amd.Manager()
    h = mgr.write(w)
    x = torch.randn(3, cols, device="cuda").to(torch.bfloat16)
    y = _product(mgr, h, x, rows)
    fin = torch.isfinite(y).all(0)
    assert fin.nonzero().flatten().tolist() == [k for k in range(rows) if k not in (5, 40, rows - 1)]
    ref = x.double() @ w.double().T
    assert torch.allclose(y[:, fin].double(), ref[:, fin], rtol=2.0 ** -7, atol=1e-3)


@pytest.mark.parametrize("cols,chunk,lane", [(520, 0, 0), (5000, 8192, 16), (40008, 0, 0)])
@pytest.mark.parametrize("scale", [2.0 ** -100, 2.0 ** -60, 2.0 ** -40, 2.0 ** 20, 2.0 ** 100])
def test_sums_have_the_range_of_fp32(scale, cols, chunk, lane):
    """Rows inside one segment, shared by two, and by as many as there can be: very small and very large sums
    come out with fp32's relative precision."""
    import neuzip_amd

    mgr = neuzip_amd.Manager(chunk_size=chunk or None, lane_symbols=lane)
    rows = 200000 // cols + 60
    gen = torch.Generator(device="cuda").manual_seed(cols)
    w = (torch.randn(rows, cols, device="cuda", generator=gen) * scale).to(torch.bfloat16)
    x = torch.randn(8, cols, device="cuda", generator=gen).to(torch.bfloat16)
    h = mgr.write(w)
    for m_rows in (1, 3, 8):
        print(f"case {rows}x{cols} {chunk}/{lane} scale={scale} rows={m_rows}", flush=True)
        with torch.no_grad():
            y = mgr.linear(h, x[:m_rows])
        _check(y, w.view(torch.int16).cpu().numpy().view(np.uint16).reshape(-1), x[:m_rows], None, 7)
    mgr._be.check()


@pytest.mark.parametrize("cols,chunk,lane", [(520, 0, 0), (5000, 8192, 16), (40008, 0, 0)])
def test_infinities_keep_their_sign(cols, chunk, lane):
    """What a sum of such values is in any order: infinite with the sign of its one infinite product, or of
    finite ones that all overflow to one side; NaN with infinities of both signs, or a NaN."""
    import neuzip_amd

    mgr = neuzip_amd.Manager(chunk_size=chunk or None, lane_symbols=lane)
    rows = 200000 // cols + 60
    w = torch.randn(rows, cols, device="cuda").to(torch.bfloat16)
    want = torch.zeros(rows)
    for k in range(0, rows, 2):  # one value, somewhere in the row
        w[k, (k * 997) % cols], want[k] = [(float("inf"),) * 2, (-float("inf"),) * 2, (float("nan"),) * 2][k // 2 % 3]
    w[1, 3], w[1, cols - 1], want[1] = float("inf"), -float("inf"), float("nan")
    w[5], want[5] = 2.0 ** 127, float("inf")
    w[7], want[7] = -2.0 ** 127, -float("inf")
    x = torch.rand(8, cols, device="cuda").to(torch.bfloat16) + 1.0
    h = mgr.write(w)
    for m_rows in (1, 8):
        with torch.no_grad():
            y = mgr.linear(h, x[:m_rows]).float().cpu()
        for got in y:
            special = want != 0
            assert torch.equal(got[special].nan_to_num(nan=0.0), want[special].nan_to_num(nan=0.0))
            assert torch.equal(got.isnan(), want.isnan()) and bool(torch.isfinite(got[~special]).all())
    mgr._be.check()


def test_linear_takes_the_product_where_it_may():
    """Manager.linear: rows of whole eights from 512 up; other lengths, traced and mapped calls and a capture
    whose accumulators would have to grow keep decompress-then-GEMM."""
    import neuzip_amd

    mgr = neuzip_amd.Manager()
    made = []
    real = mgr._be._product
    mgr._be._product = lambda fn, names, *a: (real(fn, names, *a), made.append(names[0]))[0]
    try:
        with torch.no_grad():
            for cols, takes in ((504, False), (520, True), (700, False), (1016, True), (1024, True)):
                w = (torch.randn(48, cols, device="cuda") * 0.02).to(torch.bfloat16)
                h = mgr.write(w)
                x = torch.randn(4, cols, device="cuda").to(torch.bfloat16)
                want = torch.nn.functional.linear(x, w)
                del made[:]
                assert torch.allclose(mgr.linear(h, x), want, rtol=2e-2, atol=2e-3)
                assert bool(made) == takes, cols
                if cols % 512 and takes:
                    del made[:]
                    mapped = torch.func.vmap(lambda r: mgr.linear(h, r))(x)
                    assert torch.allclose(mapped, want, rtol=2e-2, atol=2e-3) and not made
                    with torch.autograd.forward_ad.dual_level():
                        t = torch.randn_like(x)
                        d = torch.autograd.forward_ad.make_dual(x, t)
                        out = torch.autograd.forward_ad.unpack_dual(mgr.linear(h, d))
                        assert torch.allclose(out.tangent, torch.nn.functional.linear(t, w), rtol=2e-2, atol=2e-3)
                    assert not made
    finally:
        del mgr._be._product
    mgr._be.check()


def test_capture_without_a_product_before_it():
    import neuzip_amd

    mgr = neuzip_amd.Manager()
    w = (torch.randn(64, 1000, device="cuda") * 0.02).to(torch.bfloat16)
    h = mgr.write(w)
    mgr.flush()
    x = torch.randn(1, 1000, device="cuda").to(torch.bfloat16)
    torch.nn.functional.linear(x, w)  # the GEMM library is ready
    mgr.read(h)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        y = mgr.linear(h, x)
    for k in range(3):
        x.copy_(torch.randn(1, 1000, device="cuda"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.allclose(y, torch.nn.functional.linear(x, w), rtol=2e-2, atol=2e-3)
    mgr._be.check()


def test_a_captured_linear_shares_nothing_with_other_calls():
    """Rows that are not whole groups: the accumulators of the fused product belong to the manager, so a
    captured call decodes and multiplies into memory of its own and can be replayed beside products on another stream."""
    import neuzip_amd

    mgr = neuzip_amd.Manager()
    cols = 1000
    ws = [(torch.randn(64, cols, device="cuda") * 0.02).to(torch.bfloat16) for _ in range(3)]
    hs = [mgr.write(w) for w in ws]
    x = torch.randn(2, cols, device="cuda").to(torch.bfloat16)
    other = torch.randn(2, cols, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        for _ in range(3):  # the three share a launch from the second time on
            eager = [mgr.linear(h, x) for h in hs]
            mgr.linear(hs[0], other)
        mgr.linear(hs[0], x)  # leaves results of the other two behind
        for w in ws:
            torch.nn.functional.linear(x, w)  # the GEMM library is ready
        torch.cuda.synchronize()
        made = []
        real = mgr._be._product
        mgr._be._product = lambda fn, names, *a: (real(fn, names, *a), made.append(names[0]))[0]
        try:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                ys = [mgr.linear(h, x) for h in hs]
            assert not made
            side = torch.cuda.Stream()
            for k in range(4):
                x.copy_(torch.randn(2, cols, device="cuda"))
                torch.cuda.synchronize()
                with torch.cuda.stream(side):
                    beside = [mgr.linear(hs[0], other) for _ in range(8)]
                graph.replay()
                torch.cuda.synchronize()
                for y, w in zip(ys, ws):
                    assert torch.allclose(y, torch.nn.functional.linear(x, w), rtol=2e-2, atol=2e-3), k
                for y in beside:
                    assert torch.allclose(y, torch.nn.functional.linear(other, ws[0]), rtol=2e-2, atol=2e-3), k
            assert made
        finally:
            del mgr._be._product
    mgr._be.check()


@pytest.mark.parametrize("cols", [1000, 1024])
def test_an_error_of_the_product_is_raised(cols):
    """... and not answered by another path: a library that fails would look like a slow one."""
    import neuzip_amd

    mgr = neuzip_amd.Manager()
    h = mgr.write((torch.randn(48, cols, device="cuda") * 0.02).to(torch.bfloat16))
    x = torch.randn(2, cols, device="cuda").to(torch.bfloat16)

    def fails(*a):
        raise RuntimeError("planted")

    mgr._be._product = fails
    with torch.no_grad(), pytest.raises(RuntimeError, match="planted"):
        mgr.linear(h, x)
    del mgr._be._product
    with torch.no_grad():
        assert torch.isfinite(mgr.linear(h, x)).all()
    mgr._be.check()
