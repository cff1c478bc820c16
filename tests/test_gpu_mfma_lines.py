"""Matrix-core operators on 384-point lines, more tiles than resident
work-groups, and 1024-point x-lines whose tile does not fit the LDS beside an
interpolation's fragments: against the oracle at the bound of
test_gpu_mfma.py, and with an infinity or a NaN, which must spoil its whole
line and no other tile."""
import numpy as np
import pytest

from oracle import Oracle
from test_gpu_mfma import row_norm

pytestmark = pytest.mark.gpu

CASES = [((384, 128, 96), "x"), ((96, 384, 128), "y"), ((128, 96, 384), "z"), ((1024, 96, 96), "x")]
ids = dict(ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))


@pytest.mark.parametrize("op", ["der{}", "der{}pv", "int{}vp"])
@pytest.mark.parametrize("dims,axis", CASES, **ids)
def test_lines(torch_cuda, dims, axis, op):
    import torch
    from x3div_amd import X3D
    name = op.format(axis)
    print(f"\n[mfma lines {dims} {name}]", flush=True)
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
@pytest.mark.parametrize("dims", [(384, 64, 32), (1024, 64, 32)], **ids)
def test_non_finite_line(torch_cuda, dims, value):
    import torch
    from x3div_amd import X3D
    ctx = X3D(*dims)
    u = torch.rand(dims[::-1], generator=torch.Generator().manual_seed(3)).cuda()
    clean, got = ctx.field32(), ctx.field32()
    ctx.apply_circ_mfma("intxvp", clean, u)
    bad = u.clone()
    bad[17, 40, 333] = float(value)
    ctx.apply_circ_mfma("intxvp", got, bad)
    assert not torch.isfinite(got[17, 40]).any()
    same = got == clean
    assert same[:17].all() and same[18:].all() and same[17, :32].all()
    ctx.close()
