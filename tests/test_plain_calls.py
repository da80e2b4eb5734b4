"""What keeps a call on torch's own operators where they were used before: an autocast region decides the
type of their results."""
import pytest

torch = pytest.importorskip("torch")


def test_a_plain_call_is_outside_of_autocast():
    from neuzip_amd.binding import _plain_call

    x = torch.ones(2, 520, dtype=torch.bfloat16)
    assert _plain_call(x)
    was = torch.is_autocast_enabled("cuda")
    torch.set_autocast_enabled("cuda", True)
    try:
        assert not _plain_call(x)
    finally:
        torch.set_autocast_enabled("cuda", was)
    assert _plain_call(x)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_products_of_any_row_length_under_autocast(dtype):
    """Rows of 520 elements, which the fused product takes outside of such a region: the region's type, and what
    the decoded weight gives in it."""
    import neuzip_amd

    mgr = neuzip_amd.Manager(precision=7)
    gen = torch.Generator(device="cuda").manual_seed(5)
    w = (torch.randn(64, 520, device="cuda", generator=gen) * 0.02).bfloat16()
    x = torch.randn(3, 520, device="cuda", generator=gen).bfloat16()
    h = mgr.write(w)
    with torch.no_grad(), torch.autocast("cuda", dtype=dtype):
        y = mgr.linear(h, x)
        ref = torch.matmul(x, w.t())
    assert y.dtype == ref.dtype == dtype
    assert torch.equal(y, ref)
