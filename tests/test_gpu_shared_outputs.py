"""Calls that give one buffer for several outputs: the outputs are written in
order, so that the last one stays, and the others come out as with buffers
apart.  On small grids the passes of buffers apart run with one work-group per
output, those of shared buffers one output after another in a work-group: the
same operations on the same values, so every comparison here is bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# all but the last split the y and z passes in FP64 and FP32 (5 resp. 7
# wavefronts per compute unit); the last runs them unsplit either way
GRIDS = [(16, 8, 24), (40, 24, 16), (64, 64, 64), (24, 80, 48), (96, 96, 96), (128, 128, 160)]
ids = dict(ids=lambda g: "x".join(map(str, g)))
# three outputs by name, and which of x, y, z each name holds in the end
PATTERNS = [("ddd", {"d": 2}), ("ded", {"d": 2, "e": 1}), ("edd", {"d": 2, "e": 0}), ("dde", {"d": 1, "e": 2})]


def context(grid, stretch=False):
    from x3div_amd import X3D
    ctx = X3D(*grid, 6.0, 5.0, 4.0)
    if stretch:
        y = np.linspace(0.0, 1.0, grid[1])
        ctx.set_stretching(1, 1.0 + 0.3 * y, 1.0 - 0.2 * y)
    return ctx


def fields(grid, count, dtype):
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(11)
    return [torch.rand(grid[::-1], dtype=torch.float64, device="cuda", generator=gen).to(dtype) for _ in range(count)]


@pytest.mark.parametrize("stretch", [False, True], ids=["uniform", "stretched"])
@pytest.mark.parametrize("grid", GRIDS, **ids)
def test_momentum_rhs(torch_cuda, grid, stretch):
    import torch
    print(f"\n[shared du {grid} stretch {stretch}]", flush=True)
    ctx = context(grid, stretch)
    u = fields(grid, 3, torch.float64)
    du = [ctx.field() for _ in range(3)]
    ctx.calculate_transeq_rhs(*du, *u)
    for names, holds in PATTERNS:
        out = {q: ctx.field() for q in "de"}
        ctx.calculate_transeq_rhs(*(out[q] for q in names), *u)
        torch.cuda.synchronize()
        for q, k in holds.items():
            assert torch.equal(out[q], du[k]), (names, q)
    ctx.close()


@pytest.mark.parametrize("form", ["f64", "f32"])
@pytest.mark.parametrize("grid", GRIDS, **ids)
def test_step_du(torch_cuda, grid, form):
    """A step whose du share a buffer (gdt = 0: u does not take their sum)."""
    import torch
    print(f"\n[shared du in a step {grid} {form}]", flush=True)
    ctx = context(grid)
    dtype = torch.float64 if form == "f64" else torch.float32
    step = ctx.step if form == "f64" else ctx.step_f32
    u0 = fields(grid, 3, dtype)
    new = lambda: torch.zeros_like(u0[0])
    du, rest = [new() for _ in range(3)], [new() for _ in range(4)]
    step(*(a.clone() for a in u0), *du, *rest, gdt=0.0)
    for names, holds in PATTERNS:
        out = {q: new() for q in "de"}
        rest2 = [new() for _ in range(4)]
        step(*(a.clone() for a in u0), *(out[q] for q in names), *rest2, gdt=0.0)
        torch.cuda.synchronize()
        for q, k in holds.items():
            assert torch.equal(out[q], du[k]), (names, q)
        for a, b in zip(rest, rest2):
            assert torch.equal(a, b), names
    ctx.close()
