"""Steps that give one buffer for several velocities: its update and its
correction run in the order x, y, z.  A group of small grids whose gradient x
pass would otherwise run with one work-group per output, and one that would
not; every comparison is bit for bit."""
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(16, 8, 24), (40, 24, 16), (64, 64, 64), (128, 128, 160)]
# buffers of ux, uy, uz
PATTERNS = ["uuu", "uuw", "uvu", "uvv"]
ids = dict(ids=lambda g: "x".join(map(str, g)) if isinstance(g, tuple) else str(g))


def setup(grid, form):
    import torch
    from x3div_amd import X3D
    ctx = X3D(*grid, 6.0, 5.0, 4.0)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(17)
    dtype = torch.float64 if form == "f64" else torch.float32
    u0 = {q: torch.rand(grid[::-1], dtype=torch.float64, device="cuda", generator=gen).to(dtype) for q in "uvw"}
    return ctx, u0, lambda: torch.zeros(grid[::-1], dtype=dtype, device="cuda")


@pytest.mark.parametrize("form", ["f64", "f32"])
@pytest.mark.parametrize("grid", GRIDS, **ids)
def test_correction_in_order(torch_cuda, grid, form):
    """gdt = 0: the step changes the velocities by the correction alone."""
    import torch
    print(f"\n[shared velocities {grid} {form}]", flush=True)
    ctx, u0, new = setup(grid, form)
    step = ctx.step if form == "f64" else ctx.step_f32
    for names in PATTERNS:
        u = {q: a.clone() for q, a in u0.items()}
        du, pp, p = [new() for _ in range(3)], new(), [new() for _ in range(3)]
        step(*(u[q] for q in names), *du, pp, *p, gdt=0.0)
        want = {q: a.clone() for q, a in u0.items()}
        for q, g in zip(names, p):
            want[q] -= g
        torch.cuda.synchronize()
        for q in names:
            assert torch.equal(u[q], want[q]), (names, q)
    ctx.close()


@pytest.mark.parametrize("form", ["f64", "f32"])
@pytest.mark.parametrize("grid", GRIDS + [(32, 24, 320), (192, 40, 160)], **ids)
def test_step_equals_its_passes(torch_cuda, grid, form):
    """A step against the same step run as ten separate passes (the timed one),
    with buffers apart and with a velocity's buffer given again: in both the
    divergence is that of the velocities as all updates have left them."""
    import torch
    print(f"\n[step and its passes {grid} {form}]", flush=True)
    ctx, u0, new = setup(grid, form)
    step, timed = (ctx.step, ctx.step_timed) if form == "f64" else (ctx.step_f32, ctx.step_timed_f32)
    # names of ux, uy, uz, dux, duy, duz
    for names in ["uvwabc"] + [p + "abc" for p in PATTERNS] + ["uvwabu"]:
        out = []
        for run in (step, timed):
            f = {q: u0[q].clone() if q in u0 else new() for q in names}
            rest = [new() for _ in range(4)]
            run(*(f[q] for q in names), *rest, gdt=1e-3)
            out.append([f[q] for q in sorted(f)] + rest)
        torch.cuda.synchronize()
        for k, (a, b) in enumerate(zip(*out)):
            assert torch.equal(a, b), (names, k)
        assert bool(torch.isfinite(out[0][-1]).all()) and float(out[0][-1].abs().max()) > 0
    ctx.close()
