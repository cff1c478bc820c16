"""The banded walk of the matrix-core operators where it can go wrong: 768-
and 1024-point lines (tiles that fill the LDS, or do not fit it), more tiles
than resident work-groups, and lines that hold an infinity or a NaN, which
must spoil their whole line, as in the dense product, and no other tile.  The
error bound is that of test_gpu_mfma.py."""
import numpy as np
import pytest

from oracle import Oracle
from test_gpu_mfma import row_norm

pytestmark = pytest.mark.gpu

CASES = [((1024, 32, 64), "x"), ((768, 64, 32), "x"), ((32, 1024, 40), "y"), ((64, 768, 16), "y"), ((32, 16, 1024), "z"),
         ((64, 32, 768), "z"), ((128, 256, 96), "x"), ((256, 128, 40), "y"), ((256, 128, 40), "x")]


@pytest.mark.parametrize("op", ["der{}", "der{}vp", "int{}pv"])
@pytest.mark.parametrize("dims,axis", CASES, ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_band_lengths(torch_cuda, dims, axis, op):
    import torch
    from x3div_amd import X3D
    name = op.format(axis)
    print(f"\n[band {dims} {name}]", flush=True)
    orc = Oracle(*dims, 1.0, 2.0, 3.0)
    u = np.asarray(orc.fields(1, 5, 0.5)[0], dtype=np.float32)
    ref = orc.apply(name, u.astype(np.float64))
    ctx = X3D(*dims, 1.0, 2.0, 3.0)
    out = ctx.field32()
    ctx.apply_circ_mfma(name, out, torch.from_numpy(u).cuda())
    err = np.abs(out.cpu().numpy().astype(np.float64) - ref).max()
    assert err < 2.0 ** -20 * row_norm(orc, name) * np.abs(u).max()
    ctx.close()


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("axis", ["x", "y", "z"])
def test_non_finite_line(torch_cuda, axis, value):
    import torch
    from x3div_amd import X3D
    dims = (128, 128, 128)
    ctx = X3D(*dims)
    u = torch.rand((128, 128, 128), generator=torch.Generator().manual_seed(3)).cuda()
    clean, got = ctx.field32(), ctx.field32()
    ctx.apply_circ_mfma(f"der{axis}", clean, u)
    bad = u.clone()
    bad[70, 65, 40] = float(value)
    ctx.apply_circ_mfma(f"der{axis}", got, bad)
    line = {"x": (70, 65), "y": (70, slice(None), 40), "z": (slice(None), 65, 40)}[axis]
    assert not torch.isfinite(got[line]).any()
    # the tiles (32 neighbouring lines) away from it are untouched
    same = (got == clean)
    if axis == "x":
        assert same[:70].all() and same[71:].all() and same[70, :64].all() and same[70, 96:].all()
    else:
        assert same[..., :32].all() and same[..., 64:].all()
    ctx.close()
