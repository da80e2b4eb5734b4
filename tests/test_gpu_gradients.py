"""A lossless compressed Linear has the gradients of the dense one, bit for bit: of its input, its weight and
its bias, at the sizes of a small step and of a training step of 8 x 1024 tokens."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("tokens", [(4, 16), (8, 1023), (8, 1024)])
@pytest.mark.parametrize("cols,rows", [(1024, 1024), (1024, 3072), (1024, 4096), (4096, 1024)])
def test_gradients_are_those_of_the_dense_linear(tokens, cols, rows):
    import neuzip_amd

    print(f"case {tokens} {cols} -> {rows}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(rows)
    dense = torch.nn.Linear(cols, rows, device="cuda", dtype=torch.bfloat16)
    twin = torch.nn.Linear(cols, rows, device="cuda", dtype=torch.bfloat16)
    twin.load_state_dict(dense.state_dict())
    mgr = neuzip_amd.Manager()
    lin = mgr.convert(torch.nn.Sequential(twin))[0]
    x = torch.randn(*tokens, cols, device="cuda", generator=gen).to(torch.bfloat16)
    # large values that cancel and leave small sums: another order of the additions shows
    n = tokens[0] * tokens[1]
    gy = torch.randn(n, rows, device="cuda", generator=gen)
    big = torch.randn(n // 3, rows, device="cuda", generator=gen) * 1024.0
    gy[: n // 3], gy[n // 3 : 2 * (n // 3)] = big, -big
    gy = gy[torch.randperm(n, device="cuda", generator=gen)].to(torch.bfloat16).view(*tokens, rows)
    for grad in (gy, gy.transpose(0, 1).contiguous().transpose(0, 1)):
        xs = [x.clone().requires_grad_(True) for _ in range(2)]
        dense.zero_grad(), setattr(lin.bias, "grad", None), setattr(lin.weight, "_gradient", None)
        a, b = dense(xs[0]), lin(xs[1])
        assert torch.equal(a, b)
        a.backward(grad), b.backward(grad)
        assert torch.equal(xs[0].grad, xs[1].grad)
        assert torch.equal(dense.bias.grad, lin.bias.grad)
        assert torch.equal(dense.weight.grad, lin.weight._gradient)
    mgr._be.check()
