"""Row gathers that decode single segments: rows inside one, across several, across chunks, of lengths
and at places that no 16-byte store fits, out of raw chunks, with normalizers."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("norm,s", [(0, 7), (0, 3), (0, 1), (0, 0), (8, 7), (64, 3)])
@pytest.mark.parametrize("rows,dim,chunk,lane,kind", [
    (1000, 512, 0, 0, "normal"),          # a row is a group
    (300, 4096, 0, 0, "normal"),          # aligned rows: one segment each, two rings
    (4096, 7, 8192, 16, "normal"),        # shorter than a lane's eight
    (500, 701, 8192, 16, "normal"),       # odd: stored element by element, two segments at most
    (200, 2056, 8192, 16, "raw"),         # four segments of 1024
    (60, 9001, 8192, 16, "normal"),       # more than a chunk of eight
    (37, 5000, 65536, 344, "normal"),     # three segments, the last of a chunk shorter
    (3, 40000, 4096, 64, "raw"),          # one segment per chunk, ten chunks per row
    (1, 1000, 0, 0, "normal"),
])
def test_rows_of_every_length_and_place(rows, dim, chunk, lane, kind, norm, s):
    import neuzip_amd

    g = torch.Generator(device="cuda").manual_seed(rows + dim)
    if kind == "raw":
        bits = torch.randint(0, 254 << 7, (rows, dim), device="cuda", generator=g)
        w = (bits | torch.randint(0, 2, (rows, dim), device="cuda", generator=g) << 15).to(torch.int16).view(torch.bfloat16)
    else:
        w = (torch.randn(rows, dim, device="cuda", generator=g) * 0.02).to(torch.bfloat16)
    mgr = neuzip_amd.Manager(precision=s, normalizer_size=norm or None, chunk_size=chunk or None, lane_symbols=lane)
    h = mgr.write(w)
    full = mgr.read(h).view(torch.int16)
    print(f"case {rows}x{dim} {chunk}/{lane} {kind} norm={norm} s={s}", flush=True)
    every = torch.arange(rows, device="cuda")
    some = torch.cat([every[torch.randperm(rows, device="cuda", generator=g)[:150]], every[-1:], every[:1], every[:1]])
    assert torch.equal(mgr._be.gather_rows(h, some, dim).view(torch.int16), full[some])
    # into memory that begins off a 16-byte boundary
    out = torch.full((some.numel() * dim + 1,), 7.0, dtype=torch.bfloat16, device="cuda")
    be = mgr._be
    assert be._L.nz_manager_gather_rows(be._h, h.encode(), some.data_ptr(), some.numel(), dim, out[1:].data_ptr(),
                                        torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out[1:].view(-1, dim).view(torch.int16), full[some]) and float(out[0]) == 7.0
    be.check()
    # rows outside the table are rows of zeros, reported once
    far = torch.tensor([0, rows, -1, rows - 1], device="cuda")
    got = be.gather_rows(h, far, dim).view(torch.int16)
    assert torch.equal(got[::3], full[far[::3]]) and not bool(got[1:3].any())
    with pytest.raises(RuntimeError, match="outside the table"):
        be.check()
    be.check()


@pytest.mark.parametrize("precision,norm", [(7, 0), (3, 64)])
def test_captured_lookups_read_the_table(precision, norm):
    """A lookup of as many rows as the table has chunks can be captured: it reads the table and indexes."""
    import neuzip_amd

    rows, cols = 4000, 512
    mgr = neuzip_amd.Manager(precision=precision, normalizer_size=norm)
    w = (torch.randn(rows, cols, device="cuda") * 0.02).to(torch.bfloat16)
    h = mgr.write(w)
    mgr.flush()
    table = mgr.read(h).clone()
    assert rows * cols // mgr._be.geometry(h)[0] < 40
    idx = torch.randint(0, rows, (40,), device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = mgr.gather_rows(h, idx)
    for k in range(4):
        idx.copy_(torch.randint(0, rows, (40,), device="cuda"))
        graph.replay()
        eager = mgr.gather_rows(h, idx)
        torch.cuda.synchronize()
        assert torch.equal(got, table[idx]) and torch.equal(eager, table[idx]), k
    mgr._be.check()
