"""The update hook hands its tensor over to a write that is held back; plans of batched reads outlive
rewrites of the same size and not others."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


class _Rate:
    def get_last_lr(self):
        return [0.5]


def _param(mgr, *shape):
    import neuzip_amd

    w = (torch.randn(*shape, device="cuda") * 0.02).to(torch.bfloat16)
    return neuzip_amd.nn.Parameter(mgr, w.clone()), w


@pytest.mark.parametrize("ahead", [True, False])
def test_held_updates_keep_their_values(ahead):
    import neuzip_amd

    mgr = neuzip_amd.Manager()
    mgr.decode_ahead = ahead
    pairs = [_param(mgr, 64 * (k + 1), 512) for k in range(5)]
    mgr.flush()
    copied = []
    for step in range(4):
        for p, w in pairs:
            g = torch.randn(*p._shape, device="cuda").to(torch.bfloat16)
            p._gradient = g
            neuzip_amd.compressed_lomo_hook(_Rate(), p)
            assert p._gradient is None and p.grad is None
            w.add_(g, alpha=-0.5)
            copied.append(len(mgr._be._held))
        junk = [torch.full((64 * 512 * 5,), 3.0, dtype=torch.bfloat16, device="cuda") for _ in range(8)]  # memory given back?
        del junk
        for p, w in pairs:
            assert torch.equal(p(), w), step
    assert max(copied) == (len(pairs) if ahead else 1)  # (a read of its own stores what is held first)
    # a caller's own tensor is still copied
    h = pairs[0][0]._handle
    t = torch.ones(64, 512, dtype=torch.bfloat16, device="cuda")
    mgr.write(t, h)
    t.zero_()
    assert bool((mgr.read(h) == 1.0).all())
    mgr._be.check()


@pytest.mark.parametrize("fill,copied", [(4, True), (64, False)])
def test_held_updates_do_not_keep_large_buffers(fill, copied):
    """A weight decoded together with its neighbours is a view of their common buffer: held as it is,
    it would keep all of it.  (``fill`` in weights: how much may be held.)"""
    import neuzip_amd

    mgr = neuzip_amd.Manager()
    pairs = [_param(mgr, 64, 512) for _ in range(24)]
    mgr.flush()
    be = mgr._be
    be.ahead_fill = fill * 64 * 512
    for step in range(4):
        for p, w in pairs:
            g = torch.randn(64, 512, device="cuda").to(torch.bfloat16)
            p._gradient = g
            neuzip_amd.compressed_lomo_hook(_Rate(), p)
            w.add_(g, alpha=-0.5)
            stores = {t.untyped_storage().data_ptr(): t.untyped_storage().nbytes() for _, t, _ in be._held}
            assert sum(stores.values()) <= 2 * 2 * be.ahead_fill, step
        if be._held and step:
            shared = any(t.untyped_storage().nbytes() > 2 * t.numel() for _, t, _ in be._held)
            assert shared != copied
    for p, w in pairs:
        assert torch.equal(p(), w)
    mgr._be.check()


def test_plans_and_sizes_follow_the_writes():
    import neuzip_amd

    mgr = neuzip_amd.Manager()
    ws = [(torch.randn(32, 512 * (k + 1), device="cuda") * 0.02).to(torch.bfloat16) for k in range(3)]
    hs = [mgr.write(w) for w in ws]

    def pass_(n=3):
        for _ in range(n):
            for h, w in zip(hs, ws):
                assert torch.equal(mgr.read(h), w)

    pass_()
    assert mgr._be._plans
    kept = dict(mgr._be._plans)
    ws[1] = ws[1] * 2
    mgr.write(ws[1], hs[1])           # as many elements: the plans hold
    assert mgr._be._plans == kept and hs[1] in mgr._be._known
    pass_()
    ws[1] = (torch.randn(8, 520, device="cuda") * 0.02).to(torch.bfloat16)
    mgr.write(ws[1], hs[1])           # fewer: everything that knew the old size is gone
    assert not any(hs[1] in key for key in mgr._be._plans) and hs[1] not in mgr._be._known
    pass_()
    ws[2] = ws[2][:4].contiguous()
    mgr.write_many([ws[2]], [hs[2]])
    pass_()
    with pytest.raises(RuntimeError):
        mgr.write(ws[0].float(), hs[0])
    pass_(1)
    mgr._be.check()
