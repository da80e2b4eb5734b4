"""Reads enqueued behind an in-place write whose outcome the host does not know yet: of records that
fitted their buffer, that outgrew it, and that a workgroup left out because it gave up waiting."""
import numpy as np
import pytest

from conftest import bf16_bits_normal, stress_bits

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _tensor(bits):
    bits = np.where((bits >> 7 & 0xFF) == 0xFF, np.uint16(0x3C00), bits)  # finite
    return torch.from_numpy(bits.view(np.int16).copy()).cuda().view(torch.bfloat16)


def _behind_work(call):
    """call() behind some milliseconds of other work on the stream -> (its result, whether it came back before that ended)"""
    done = torch.cuda.Event()
    torch.cuda._sleep(40_000_000)
    done.record()
    out = call()
    return out, not done.query()


def _same(a, b):
    return torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("spins", [1 << 15, 0])  # none: workgroups give up at their first look
@pytest.mark.parametrize("norm,s", [(0, 7), (64, 3)])
def test_read_of_a_write_that_is_still_running(spins, norm, s):
    import neuzip_amd
    from neuzip_amd import _lib

    mgr = neuzip_amd.Manager(precision=s, normalizer_size=norm or None)
    mgr.decode_ahead = False
    n = 41 * 131072 + 1024
    flat = torch.full((n,), 0.5, dtype=torch.bfloat16, device="cuda")
    tight = _tensor(bf16_bits_normal(n, seed=3))
    noisy = _tensor(stress_bits(n // 1024, 1024, seed=4))
    odd = [_tensor(bf16_bits_normal(k, seed=k)) for k in (1000, 2_000_003)]
    ref = neuzip_amd.Manager(precision=s, normalizer_size=norm or None)  # what a value reads back as

    def stored(w):
        return ref.read(ref.write(w, "x"))

    first = [flat, tight, *odd]
    hs = [mgr.write(w) for w in first]
    mgr.flush()
    try:
        _lib.load().nz_set_lookback_spins(spins)
        # a first write outgrows the first buffer, the next ones go back and forth in the larger one
        for turn, new in enumerate(([noisy, tight, *odd], [flat, noisy, *[-w for w in odd]], [tight, tight, *odd])):
            print(f"case spins={spins} norm={norm} turn={turn}", flush=True)

            def call():
                mgr.write_many(new, hs)
                single = [mgr.read(h) for h in hs]
                outs = [torch.empty(w.numel(), dtype=torch.bfloat16, device="cuda") for w in new]
                mgr._be.read_batch(mgr._be.batch_plan(hs), outs)
                return single, outs

            (single, outs), ahead = _behind_work(call)
            assert ahead == (turn > 0)  # the first time a read comes this soon it waits
            want = [stored(w) for w in new]
            for a, b, w in zip(single, outs, want):
                assert _same(a, w) and _same(b, w)
            for h, w in zip(hs, want):  # ... and once the host has looked at the outcome
                assert _same(mgr.read(h), w)
        # many writes and reads with no look at any outcome in between but the manager's own
        def many():
            got = []
            for k in range(6):
                mgr.write_many([(noisy, flat, tight)[k % 3]], hs[:1])
                got.append(mgr.read(hs[0]))
            return got

        got, _ = _behind_work(many)
        for k, r in enumerate(got):
            assert _same(r, stored((noisy, flat, tight)[k % 3])), k
    finally:
        _lib.load().nz_set_lookback_spins(1 << 15)
    mgr._be.check()
    mgr.trim()
    assert _same(mgr.read(hs[0]), stored(tight))


def test_read_on_another_stream_waits_for_the_write():
    import neuzip_amd

    mgr = neuzip_amd.Manager()
    ws = [(torch.randn(1 << 20, device="cuda") * 0.02).to(torch.bfloat16) for _ in range(2)]
    h = mgr.write(ws[0])
    mgr.flush()
    side = torch.cuda.Stream()
    for k in range(4):
        torch.cuda._sleep(2_000_000)
        mgr.write_many([ws[k % 2]], [h])
        a = mgr.read(h)
        with torch.cuda.stream(side):
            b = mgr.read(h)
        side.synchronize()
        assert torch.equal(a, ws[k % 2]) and torch.equal(b, ws[k % 2])
    torch.cuda.current_stream().wait_stream(side)
    mgr._be.check()
