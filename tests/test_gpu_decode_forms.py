"""Both forms of the decode step: launches of up to one workgroup (chunk) per compute unit, 256 on
a whole GPU, read one prepared entry per step from a wide ring; larger ones the slot table and the
word in turn for dense output, and one entry per step from a narrow ring for products
(tests/test_launch_forms.py pins the rule).  Every kernel that decodes is run with as many chunks as
the line and with one more: reads at every precision, with normalizers, of several tensors at once
and of corrupt containers, row gathers, and products with one to eight activation rows."""
import ctypes

import numpy as np
import pytest

from conftest import bf16_bits_normal, closed_form_recon, stress_bits
from test_gpu_fused_gemv import _check, _gemv
from test_gpu_parity import gpu_decode, gpu_encode

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CHUNK, LANE = 8192, 16  # small chunks: eight wavefronts of 16 symbols per lane
LINE = [256, 257]


def _bits(kind, n):
    rng = np.random.default_rng(n)
    low = rng.integers(0, 1 << 16, n, dtype=np.uint32) & 0x807F
    if kind == "normal":
        return bf16_bits_normal(n, seed=n & 0xFFFF)
    if kind == "constant":  # hardly a word in the whole record
        exps = np.full(n, 120)
    elif kind == "wide":  # 6 bits a symbol: three words per lane and group of eight
        exps = rng.integers(60, 124, n)
    else:  # runs of rare symbols (8 bits each at chunks of 8192, 11 at 65536) in every lane at once,
        # between runs that take nothing
        exps = np.full(n, 120)
        at = np.arange(n) // 4096 % 61 == 7
        exps[at] = rng.integers(0, 120, int(at.sum()))
    return (low | (exps.astype(np.uint32) << 7)).astype(np.uint16)


def _records(comp, n, chunk, lane):
    """Byte offsets of the segment records (and of their end) in a container."""
    spc = -(-chunk // (64 * lane))
    full, rest = divmod(n, chunk)
    segs = full * spc + -(-rest // (64 * lane))
    rec_off = (64 + 4 * (segs + 1) + 15) & ~15
    return rec_off + 4 * comp[64:64 + 4 * (segs + 1)].view(np.uint32).astype(np.int64), spc


def _coded_chunks(comp, n, chunk, lane):
    at, spc = _records(comp, n, chunk, lane)
    return int(np.count_nonzero(comp[at[:-1:spc]] != 0xFF))


def _dev(bits, *shape):
    return torch.from_numpy(bits.view(np.int16).copy()).cuda().view(torch.bfloat16).view(*shape)


def _host(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16).reshape(-1)


@pytest.mark.parametrize("kind", ["normal", "constant", "wide", "bursts"])
@pytest.mark.parametrize("chunk,lane,n", [(8192, 16, 256 * 8192), (8192, 16, 256 * 8192 + 1),
                                          (65536, 128, 256 * 65536), (65536, 128, 256 * 65536 + 1),
                                          (32768, 128, 600_011), (131072, 256, 1_000_003)])
def test_decode_forms(kind, chunk, lane, n):
    """Lossless, so the result is the input bit for bit; of full chunks all are coded, none stored raw."""
    bits = _bits(kind, n)
    print(f"case {kind} chunk={chunk} lane={lane} n={n}", flush=True)
    comp, packed = gpu_encode(bits, 7, chunk, lane)
    assert _coded_chunks(comp.cpu().numpy(), n, chunk, lane) >= n // chunk
    rc, out = gpu_decode(comp, packed, n, 7, chunk, lane)
    assert rc == 0 and np.array_equal(out, bits)


@pytest.mark.parametrize("chunks", LINE)
@pytest.mark.parametrize("s,norm", [(3, 0), (1, 0), (0, 0), (7, 4), (7, 64), (3, 4), (3, 64), (0, 8)])
def test_lossy_and_normalized_reads(oracle, s, norm, chunks):
    n = CHUNK * (chunks - 1) + 4099
    bits = bf16_bits_normal(n, seed=s + norm)
    print(f"case s={s} norm={norm} chunks={chunks}", flush=True)
    comp, packed, *nb = gpu_encode(bits, s, CHUNK, LANE, norm)
    rc, out = gpu_decode(comp, packed, n, s, CHUNK, LANE, norm_size=norm, norm=nb[0] if nb else None)
    want = oracle.reconstruct_normalized(bits, s, norm) if norm else closed_form_recon(bits, s)
    assert rc == 0 and np.array_equal(out, want)


@pytest.mark.parametrize("chunks", LINE)
def test_corrupt_containers_are_reported(oracle, chunks):
    n = CHUNK * chunks
    bits = bf16_bits_normal(n, seed=chunks)
    comp, packed = gpu_encode(bits, 7, CHUNK, LANE)
    host, frac = comp.cpu().numpy(), packed.cpu().numpy()
    at, spc = _records(host, n, CHUNK, LANE)
    # (a record's states end below its byte 288; its last words reach only carried bits, which nothing checks)
    for what, pos in (("words of the first record", at[0] + 330), ("words of a middle record", at[at.size // 2] + 300),
                      ("words of the last record", at[-2] + 300), ("states of a middle record", at[at.size // 2 + 1] + 40)):
        bad = host.copy()
        bad[pos] ^= 0x5A
        print(f"case {what} chunks={chunks}", flush=True)
        assert oracle.decompress_bf16(bad, frac, n, 7)[0] != 0
        assert gpu_decode(torch.from_numpy(bad).cuda(), packed, n, 7, CHUNK, LANE)[0] == -6
    bad = host.copy()
    bad[64 + 4 * spc * (chunks - 1):][:8] = 0xFF  # the last chunk's directory entries
    print(f"case directory chunks={chunks}", flush=True)
    assert gpu_decode(torch.from_numpy(bad).cuda(), packed, n, 7, CHUNK, LANE)[0] == -6


@pytest.mark.parametrize("chunks", LINE)
@pytest.mark.parametrize("s,norm", [(7, 0), (3, 0), (1, 0), (3, 64), (0, 8)])
def test_several_tensors_in_one_launch(oracle, s, norm, chunks):
    import neuzip_amd

    mgr = neuzip_amd.Manager(precision=s, normalizer_size=norm, chunk_size=CHUNK, lane_symbols=LANE)
    sizes = [100 * CHUNK, 77 * CHUNK - 5, (chunks - 177) * CHUNK - 4001]
    bits = [bf16_bits_normal(n, seed=i) for i, n in enumerate(sizes)]
    hs = [mgr.write(_dev(b, b.size)) for b in bits]
    outs = [torch.zeros(n, dtype=torch.bfloat16, device="cuda") for n in sizes]
    print(f"case s={s} norm={norm} chunks={chunks}", flush=True)
    mgr._be.read_batch(mgr._be.batch_plan(hs), outs)
    for b, o in zip(bits, outs):
        want = oracle.reconstruct_normalized(b, s, norm) if norm else closed_form_recon(b, s)
        assert np.array_equal(_host(o), want)
    mgr._be.check()


@pytest.mark.parametrize("s,norm", [(7, 0), (3, 0), (1, 0), (3, 64), (0, 8)])
@pytest.mark.parametrize("rows,dim,count", [
    (30_000, 64, 256), (30_000, 64, 257),      # rows inside a chunk: one workgroup per row
    (30_000, 24, 128), (30_000, 24, 129),      # rows straddle chunks: two workgroups per row
])
def test_row_gathers(oracle, rows, dim, count, s, norm):
    import neuzip_amd

    mgr = neuzip_amd.Manager(precision=s, normalizer_size=norm, chunk_size=CHUNK, lane_symbols=LANE)
    bits = bf16_bits_normal(rows * dim, seed=dim)
    h = mgr.write(_dev(bits, rows, dim))
    full = _dev(oracle.reconstruct_normalized(bits, s, norm) if norm else closed_form_recon(bits, s), rows, dim)
    idx = torch.randint(0, rows, (count,), generator=torch.Generator().manual_seed(count))
    idx[0], idx[-1] = rows - 1, 0
    print(f"case rows={rows} dim={dim} count={count} s={s} norm={norm}", flush=True)
    assert torch.equal(mgr._be.gather_rows(h, idx.cuda(), dim), full[idx.cuda()])
    mgr._be.check()


@pytest.mark.parametrize("chunks", LINE)
@pytest.mark.parametrize("s", [7, 3, 1, 0])
@pytest.mark.parametrize("m_rows", [1, 2, 3, 8])
def test_products(m_rows, s, chunks):
    """Rows of 1536 weights straddle the segments of 1024; one to eight activation rows, each the
    bits of the one-row call and within its tolerance of the fp64 product."""
    import neuzip_amd

    cols = 1536
    rows = CHUNK * chunks // cols
    assert -(-rows * cols // CHUNK) == chunks
    mgr = neuzip_amd.Manager(precision=s, chunk_size=CHUNK, lane_symbols=LANE)
    bits = bf16_bits_normal(rows * cols, seed=chunks + s)
    h = mgr.write(_dev(bits, rows, cols))
    assert mgr._be.geometry(h) == (CHUNK, LANE)
    g = torch.Generator(device="cuda").manual_seed(m_rows)
    x = torch.randn(m_rows, cols, device="cuda", generator=g).to(torch.bfloat16)
    bias = torch.randn(rows, device="cuda", generator=g).to(torch.bfloat16)
    out = torch.full((m_rows, rows), 7.0, dtype=torch.bfloat16, device="cuda")
    print(f"case rows={m_rows} s={s} chunks={chunks}", flush=True)
    mgr._be.gemv_batch((ctypes.c_char_p * 1)(h.encode()), x if m_rows > 1 else x[0], [bias],
                       [out if m_rows > 1 else out[0]], m_rows)
    for m in range(m_rows):
        (one,) = _gemv(mgr, [h], x[m].contiguous(), [bias])
        assert torch.equal(one.view(torch.int16), out[m].view(torch.int16))
        _check(out[m], bits, x[m], bias, s)
    mgr._be.check()


@pytest.mark.parametrize("chunks", LINE)
@pytest.mark.parametrize("s", [7, 3])
def test_products_with_normalizers(oracle, s, chunks):
    import neuzip_amd

    cols = 1536
    rows = CHUNK * chunks // cols
    mgr = neuzip_amd.Manager(precision=s, normalizer_size=64, chunk_size=CHUNK, lane_symbols=LANE)
    bits = stress_bits(rows, cols, seed=chunks + s)
    bits = np.where(((bits >> 7) & 0xFF) == 0xFF, np.uint16(0x3C00), bits)  # finite
    h = mgr.write(_dev(bits, rows, cols))
    x = torch.randn(cols, device="cuda", generator=torch.Generator(device="cuda").manual_seed(s)).to(torch.bfloat16)
    print(f"case s={s} chunks={chunks}", flush=True)
    (y,) = _gemv(mgr, [h], x, None)
    # the reconstruction is what the product multiplies: lossless from here on
    _check(y, oracle.reconstruct_normalized(bits, s, 64), x, None, 7)
    mgr._be.check()


@pytest.mark.parametrize("kind", ["normal", "wide", "bursts"])
@pytest.mark.parametrize("chunk,lane,cols", [(131072, 256, 4096),  # from six rows on with staged activations
                                             (65536, 128, 1536)])  # rows straddle the segments of 8192
def test_products_that_take_many_words(kind, chunk, lane, cols):
    """More than 256 workgroups: the narrow ring.  It is looked at once per group of 512 symbols, when
    at least 129 words are left in it; a group that takes more ("wide": 192, "bursts": up to 350) refills it inside."""
    import neuzip_amd

    rows = 257 * chunk // cols + 1
    n = rows * cols
    bits = _bits(kind, n)
    mgr = neuzip_amd.Manager(chunk_size=chunk, lane_symbols=lane)
    w = _dev(bits, rows, cols)
    h = mgr.write(w)
    assert _coded_chunks(mgr._be.export(h)[0].numpy(), n, chunk, lane) >= n // chunk > 256
    g = torch.Generator(device="cuda").manual_seed(cols)
    x = torch.randn(8, cols, device="cuda", generator=g).to(torch.bfloat16)
    want = x.double() @ w.double().t()
    # a bf16 rounding of the result; fp32 sums; partial sums of a shared row resolved to 2^-40
    tol = 2.0 ** -8 * want.abs() + 1e-5 * (x.double().abs() @ w.double().abs().t()) + 2.0 ** -36
    ones = torch.stack([_gemv(mgr, [h], x[m].contiguous(), None)[0] for m in range(8)])
    assert bool(((ones.double() - want).abs() <= tol).all())
    for m_rows in (2, 5, 6, 8):
        print(f"case {kind} chunk={chunk} cols={cols} rows={m_rows}", flush=True)
        out = torch.full((m_rows, rows), 7.0, dtype=torch.bfloat16, device="cuda")
        mgr._be.gemv_batch((ctypes.c_char_p * 1)(h.encode()), x[:m_rows].contiguous(), [None], [out], m_rows)
        assert torch.equal(out.view(torch.int16), ones[:m_rows].view(torch.int16)), m_rows
    mgr._be.check()
