"""Passes of small grids run with one work-group per output; a gradient whose
outputs share a buffer runs them in order.  Both have to give the same bits:
the same operations on the same values."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(16, 8, 24), (40, 24, 16), (64, 64, 64), (96, 96, 96), (128, 128, 128)],
                         ids=lambda g: "x".join(map(str, g)))
def test_gradient_outputs_apart_or_in_one_buffer(torch_cuda, grid):
    import torch
    from x3div_amd import X3D
    print(f"\n[split {grid}]", flush=True)
    ctx = X3D(*grid, 6.0, 5.0, 4.0)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(11)
    pp = torch.rand(grid[::-1], dtype=torch.float64, device="cuda", generator=gen)
    p = [ctx.field() for _ in range(3)]
    ctx.gradp(*p, pp)
    one = ctx.field()
    ctx.gradp(one, one, one, pp)
    torch.cuda.synchronize()
    assert torch.equal(one, p[2])
    for a in p:
        assert float(a.abs().max()) > 0
    ctx.close()
