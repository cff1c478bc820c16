"""Non-periodic first derivatives and in-place Thomas sweeps at every chunk
length that the line kernels are built for (x 6-16 points, y and z 8-16), at
the lengths where a chunking can go wrong: the shortest line of a chunk
length, the one with the most padding (whole chunks of it), and one whose last
two rows lie in different chunks.  99 lines, so that the last wavefront or
work-group is partly filled.  Against the oracle at the bar of the other
non-periodic tests, 1e-12 of the result's maximum."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

# points per chunk: shortest line, most padding, last two rows apart
X = {6: (11, 321, 379), 7: (13, 385, 442), 8: (8, 449, 505), 9: (9, 513, 568), 10: (10, 577, 631), 11: (641, 694),
     12: (705, 757), 13: (769, 820), 14: (833, 883), 15: (897, 946), 16: (961, 1009)}
YZ = {8: (8,), 9: (9, 513, 568), 10: (10, 577, 631), 11: (11, 641, 694), 12: (12, 705, 757), 13: (13, 769, 820),
      14: (14, 833, 883), 15: (15, 897, 946), 16: (16, 961, 1009)}
LINES = [(axis, n) for axis, t in (("x", X), ("y", YZ), ("z", YZ)) for ns in t.values() for n in ns]


@pytest.mark.parametrize("axis,n", LINES, ids=lambda v: str(v))
def test_chunk_lengths(torch_cuda, axis, n):
    import torch
    from x3div_amd import X3D
    grid = {"x": (n, 9, 11), "y": (9, n, 11), "z": (9, 11, n)}[axis]
    u = np.random.default_rng(n).standard_normal(grid[::-1])
    ud = torch.from_numpy(u).cuda()
    for bc in ((1, 1), (1, 2), (2, 1), (2, 2)):
        print(f"\n[np chunks {axis} {n} bc {bc}]", flush=True)
        ctx = X3D(*grid, 1.0, 2.0, 3.0, ncl1=(bc[0],) * 3, ncln=(bc[1],) * 3)
        length = {"x": 1.0, "y": 2.0, "z": 3.0}[axis]
        tb = oracle.np_tables(n, length / (n - 1), *bc)
        for npaire, name, p in ((0, f"der{axis}", ""), (1, f"der{axis}p", "p")):
            t = ctx.field()
            getattr(ctx, f"der{axis}")(t, ud, name)
            ref = oracle.der_np(u, axis, length, *bc, npaire)
            assert np.abs(t.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max(), (bc, name)
            tt = ud.clone()
            getattr(ctx, f"{axis}thomas")(tt, name)
            ref = u.copy()
            getattr(oracle.lib(False), f"orc_{axis}thomas_12")(
                oracle._p(ref), *(oracle._p(tb[k + p]) for k in "fsw"), *grid)
            assert np.abs(tt.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max(), (bc, name, "thomas")
        ctx.close()
