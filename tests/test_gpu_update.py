"""int_time and cor_vel (o_k = g a_k + o_k, o_k = o_k - a_k for k = x, y, z in
this order) where one launch for the three components could go wrong: a buffer
given for two components or as another's operand, overlapping buffers, odd
point counts and bases that are not 16-byte aligned.  Small whole numbers and
g = 1/2: every sum is exact, so the results are equal to numpy's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (grid, boundary codes): even and odd point counts (5049 and 1), one block and many
GRIDS = [((16, 8, 24), 0), ((33, 17, 9), 2), ((128, 64, 96), 0), ((129, 65, 33), 1)]
# operands by name: ux, uy, uz, then the three added or subtracted
CALLS = {"apart": "ABCDEF", "one output": "AAADEF", "two outputs": "ABADEF", "one input": "ABCDDD", "input of the next": "ABCDAE",
         "input of the one before": "ABCBDE", "own input": "ABCABC", "all one": "AAAAAA"}


def check(grid, bc, views, call, tag):
    """views: {name: (offset, host values)} into one allocation of 8-byte words."""
    import torch
    from x3div_amd import X3D
    nx, ny, nz = grid
    n = nx * ny * nz
    ctx = X3D(nx, ny, nz, 1.0, 1.0, 1.0, ncl1=(bc,) * 3, ncln=(bc,) * 3)
    rng = np.random.default_rng(5)
    host = rng.integers(-8, 9, max(views.values()) + n).astype(np.float64)
    for sub in (False, True):
        dev = torch.from_numpy(host.copy()).cuda()
        want = host.copy()
        f = [dev[views[q]:views[q] + n].view(nz, ny, nx) for q in call]
        w = [want[views[q]:views[q] + n] for q in call]
        print(f"\n[update {grid} {tag} {'cor_vel' if sub else 'int_time'}]", flush=True)
        if sub:
            ctx.cor_vel(*f)
        else:
            ctx.int_time(*f, 0.5)
        for k in range(3):
            a = w[k + 3].copy()
            w[k][:] = w[k] - a if sub else 0.5 * a + w[k]
        torch.cuda.synchronize()
        assert np.array_equal(dev.cpu().numpy(), want), (tag, sub)
    ctx.close()


@pytest.mark.parametrize("call", CALLS, ids=lambda c: c.replace(" ", "-"))
@pytest.mark.parametrize("grid,bc", GRIDS, ids=lambda g: "x".join(map(str, g)) if isinstance(g, tuple) else f"ncl{g}")
def test_shared_buffers(torch_cuda, grid, bc, call):
    n = int(np.prod(grid))
    step = n + n % 2  # every base 16-byte aligned
    check(grid, bc, {q: k * step for k, q in enumerate("ABCDEF")}, CALLS[call], call)


@pytest.mark.parametrize("grid,bc", GRIDS, ids=lambda g: "x".join(map(str, g)) if isinstance(g, tuple) else f"ncl{g}")
def test_unaligned_and_overlapping(torch_cuda, grid, bc):
    n = int(np.prod(grid))
    step = n + n % 2
    # one base off by a word, then all of them
    for off in ([0, 0, 1, 0, 0, 0], [1] * 6):
        check(grid, bc, {q: k * (step + 2) + off[k] for k, q in enumerate("ABCDEF")}, "ABCDEF", f"unaligned {off}")
    # B starts inside A, and E (the second operand) inside A as well
    check(grid, bc, {"A": 0, "B": n // 2, "C": 2 * step, "D": 3 * step, "E": 4 * step, "F": 5 * step}, "ABCDEF", "outputs overlap")
    check(grid, bc, {"A": 0, "B": 6 * step, "C": 2 * step, "D": 3 * step, "E": n // 4, "F": 5 * step}, "ABCDEF", "input in an output")
