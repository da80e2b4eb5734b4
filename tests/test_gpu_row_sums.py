"""Sums over the rows of a bf16 matrix, and the bias gradient that goes by them."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("rows,cols", [
    (1, 8), (3, 512), (4, 520), (31, 72), (32, 64), (33, 504), (64, 1024), (1000, 136), (4097, 1032), (20011, 8),
    (8192, 1024), (300, 40000), (70000, 264),
])
def test_row_sums(rows, cols):
    from neuzip_amd import _lib

    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, cols, device="cuda", generator=g).to(torch.bfloat16)
    guard = 64
    scratch = torch.full((lib.nz_row_sums_bytes(rows, cols) // 4 + guard,), 7.0, device="cuda")
    out = torch.full((cols + guard,), 7.0, dtype=torch.bfloat16, device="cuda")
    print(f"case {rows}x{cols}", flush=True)
    assert lib.nz_row_sums(x.data_ptr(), rows, cols, scratch.data_ptr(), out.data_ptr(),
                           torch.cuda.current_stream().cuda_stream) == 0
    assert bool((out[cols:] == 7.0).all()) and bool((scratch[-guard:] == 7.0).all())
    want = x.double().sum(0)
    # Half a unit in the last place of the result: bf16 has 8 significant bits, so that is 2^-8 of the power of two
    # at or below it, at most 2^-8 of the result.  And 2^-24 of the magnitudes per addition of a chain: a lane's
    # rows / 4 / workgroups of at most 160 for these, 4, parts / 16 and 16.
    tol = 2.0 ** -8 * want.abs() + 2.0 ** -16 * x.double().abs().sum(0)
    assert bool(((out[:cols].double() - want).abs() <= tol).all())
    # one value that is not finite stays in its column
    x[rows // 2, 5] = float("inf")
    assert lib.nz_row_sums(x.data_ptr(), rows, cols, scratch.data_ptr(), out.data_ptr(),
                           torch.cuda.current_stream().cuda_stream) == 0
    assert torch.isinf(out[:cols]).nonzero().flatten().tolist() == [5]
    assert lib.nz_row_sums(x.data_ptr(), rows, cols + 4, scratch.data_ptr(), out.data_ptr(), None) == _lib.ERR_ARG
    assert lib.nz_row_sums(x.data_ptr() + 2, rows, cols, scratch.data_ptr(), out.data_ptr(), None) == _lib.ERR_ALIGN


def test_bias_gradient_of_large_steps():
    """By the row sums where the gradient is a large contiguous bf16 matrix and nothing is recorded;
    by torch's sum otherwise."""
    import neuzip_amd

    dense = torch.nn.Linear(1024, 1024, device="cuda", dtype=torch.bfloat16)
    b = dense.bias.data.clone()
    w = dense.weight.data.clone()
    lin = neuzip_amd.Manager().convert(torch.nn.Sequential(dense))[0]
    for rows in (8192, 8191):  # 8 M elements, and less
        x = torch.randn(rows, 1024, device="cuda", dtype=torch.bfloat16).requires_grad_(True)
        gy = torch.randn(rows, 1024, device="cuda", dtype=torch.bfloat16)
        for grad in (gy, gy.t().contiguous().t()):  # the second one is not contiguous
            lin.bias.grad = None
            lin(x).backward(grad)
            want = gy.double().sum(0)
            tol = 2.0 ** -8 * want.abs() + 2.0 ** -16 * gy.double().abs().sum(0)
            assert bool(((lin.bias.grad.double() - want).abs() <= tol).all())
    # a backward pass that is recorded itself
    x = torch.randn(8192, 1024, device="cuda", dtype=torch.bfloat16).requires_grad_(True)
    gy = torch.randn(8192, 1024, device="cuda", dtype=torch.bfloat16).requires_grad_(True)
    (gb,) = torch.autograd.grad(lin(x), lin.bias, gy, create_graph=True)
    assert gb.requires_grad
    (back,) = torch.autograd.grad(gb.float().sum(), gy)
    assert torch.equal(back, torch.ones_like(back))
    assert torch.equal(b, lin.bias.data) and torch.equal(lin.weight(), w)
