"""Decodes and products of so few chunks that several workgroups share each: every split of a chunk's
segments, chunks of one to eight, whole and cut short, compressible and raw."""
import ctypes

import numpy as np
import pytest

from conftest import bf16_bits_normal

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("segs", [1, 2, 3, 5, 7, 8])
@pytest.mark.parametrize("chunks", [1, 2, 32, 33, 64, 65, 128, 129])
def test_chunks_shared_by_workgroups(segs, chunks):
    import neuzip_amd

    chunk = 1024 * segs
    n = chunk * chunks
    g = torch.Generator(device="cuda").manual_seed(segs * 1000 + chunks)
    mgr = neuzip_amd.Manager(chunk_size=chunk, lane_symbols=16)
    print(f"case {chunks} chunks of {segs} segments", flush=True)
    ws = []
    for cut in (0, 512, 777, 1024 * (segs // 2) + 512):
        w = torch.from_numpy(bf16_bits_normal(n, seed=cut).view(np.int16).copy()).cuda().view(torch.bfloat16)
        # a chunk in the middle that does not compress
        raw = torch.randint(0, 254 << 7, (chunk,), device="cuda", generator=g).to(torch.int16).view(torch.bfloat16)
        w[chunk * (chunks // 2):][:chunk] = raw
        if n - cut > 0:
            ws.append(w[:n - cut].contiguous())
    hs = [mgr.write(w) for w in ws]
    for h, w in zip(hs, ws):
        assert mgr._be.geometry(h) == (chunk, 16)
        assert torch.equal(mgr._be.read(h).view(torch.int16), w.view(torch.int16))
    outs = [torch.empty_like(w) for w in ws[:2]]
    mgr._be.read_batch(mgr._be.batch_plan(hs[:2]), outs)
    for o, w in zip(outs, ws):
        assert torch.equal(o.view(torch.int16), w.view(torch.int16))
    # products: rows of 512, and (where there are that many elements) rows that four segments share
    for cols in (512, 3584):
        if n % cols or n // cols < 1:
            continue
        w = (torch.randn(n, device="cuda", generator=g) * 0.02).to(torch.bfloat16)
        h = mgr.write(w)
        x = torch.randn(8, cols, device="cuda", generator=g).to(torch.bfloat16)
        names = (ctypes.c_char_p * 1)(h.encode())
        ref = x.double() @ w.view(-1, cols).double().T
        tol = 2.0 ** -8 * ref.abs() + 1e-5 * (x.double().abs() @ w.view(-1, cols).double().abs().T) + 2.0 ** -36
        for rows in (1, 8):
            y = torch.empty(rows, n // cols, dtype=torch.bfloat16, device="cuda")
            mgr._be.gemv_batch(names, x[:rows].contiguous(), None, [y], rows)
            assert bool(((y.double() - ref[:rows]).abs() <= tol[:rows]).all())
    mgr._be.check()
