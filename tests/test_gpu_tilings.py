"""GPU parity of the step over the line tilings that the chunk-length rule
picks: every 3- and 5-smooth length in each direction, on grids around the
sizes where the chunk caps change (8 and 16 points in FP64; 8, 16 and 32 in
FP32), against the CPU oracle at the step's bars: 1e-12 in FP64 (the pressure
1e-11), the batch tests' FP32 bounds on velocity and pressure, and BFP32
within 1e-6."""
import numpy as np
import pytest

from oracle import Oracle

pytestmark = pytest.mark.gpu

GRIDS = [(16, 16, 16), (32, 32, 32), (24, 320, 160), (40, 384, 80), (48, 96, 192), (80, 24, 384), (96, 192, 48),
         (160, 40, 96), (192, 80, 40), (320, 48, 24), (384, 160, 24), (16, 48, 320), (64, 64, 64), (80, 80, 80)]
# 32-point FP32 chunks: 10 and 5 per line (2 and 1 chunk groups)
GRIDS32 = [(32, 320, 320), (160, 160, 160)]
L = (2 * np.pi, 1.5 * np.pi, 2.5 * np.pi)


def relerr(a, b):
    a = np.asarray(a, dtype=np.float64)
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


@pytest.mark.parametrize("grid", GRIDS + GRIDS32, ids=lambda g: "x".join(map(str, g)))
def test_step_over_tilings(torch_cuda, grid):
    import torch
    from x3div_amd import X3D, X3DError
    print(f"\n[tilings {grid}]", flush=True)
    orc = Oracle(*grid, *L)
    u0 = orc.fields(2, 99, 0.0)
    u, du, pp, g = orc.step(*u0, gdt=1e-3)
    ctx = X3D(*grid, *L)
    dev = [torch.from_numpy(a.copy()).cuda() for a in u0]
    if grid in GRIDS:
        f = [a.clone() for a in dev] + [ctx.field() for _ in range(7)]
        ctx.step(*f, gdt=1e-3)
        for a, r in zip(f[:6], list(u) + list(du)):
            assert relerr(a.cpu().numpy(), r) < 1e-12
        for a, r in zip(f[6:], [pp] + list(g)):
            assert relerr(a.cpu().numpy(), r) < 1e-11
    f = [a.float() for a in dev] + [ctx.field32() for _ in range(7)]
    ctx.step_f32(*f, gdt=1e-3)
    for a, r in zip(f[:3], u):
        assert relerr(a.cpu().numpy(), r) < 2e-4
    assert relerr(f[6].cpu().numpy(), pp) < 2e-3
    if grid in GRIDS and grid[0] % 16 == 0:
        f = [ctx.bfp_empty() for _ in range(10)]
        if 320 in grid[1:]:  # not tiled with whole 16-line rows by a power of two of chunks: refused
            with pytest.raises(X3DError, match="UNSUPPORTED"):
                ctx.step_bfp(*f, gdt=1e-3)
            return
        for q, a in zip(f, dev):
            ctx.bfp_encode(q, a)
        ctx.step_bfp(*f, gdt=1e-3)
        t = ctx.field()
        for q, r in zip(f[:6], list(u) + list(du)):
            ctx.bfp_decode(t, q)
            assert relerr(t.cpu().numpy(), r) < 1e-6
    ctx.close()
