"""Every pass of a small grid that runs with one work-group per output, against
the same passes of a batch of one grid, whose kernels run the outputs one after
another on the same tilings: the same operations on the same values, so all ten
fields of a step are equal bit for bit.  FP64 grids are those whose Poisson the
batch solves as a single grid does (24- and 40-point x-lines); on others the
pressure's last transform is another kernel, and the momentum alone is compared."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SMALL = [(40, 24, 16), (24, 80, 48), (40, 64, 96), (24, 160, 64)]
GRIDS = SMALL + [(16, 8, 24), (64, 64, 64), (96, 96, 96), (128, 128, 160)]


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "x".join(map(str, g)))
def test_step_equals_batch_of_one(torch_cuda, grid, precision):
    import torch
    from x3div_amd import X3D, X3DBatch
    print(f"\n[split bits {grid} precision {precision}]", flush=True)
    rng = np.random.default_rng(3)
    u = [rng.standard_normal(grid[::-1]).astype(np.float64 if precision == 8 else np.float32) for _ in range(3)]
    batch = X3DBatch([grid], precision=precision)
    for name, a in zip(batch.FIELDS, u):
        batch.put(0, name, a)
    batch.step(gdt=1e-3)
    ctx = X3D(*grid, *(2 * np.pi,) * 3)
    f = [torch.from_numpy(a).cuda() for a in u] + [ctx.field() if precision == 8 else ctx.field32() for _ in range(7)]
    (ctx.step if precision == 8 else ctx.step_f32)(*f, gdt=1e-3)
    torch.cuda.synchronize()
    for name, a in zip(batch.FIELDS, f):
        if precision == 4 or grid in SMALL or name.startswith("d"):
            assert np.array_equal(a.cpu().numpy(), batch.get(0, name)), name
    batch.close()
    ctx.close()
