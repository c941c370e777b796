"""GPU: the flow update's choices by grid size against each other.

The momentum kernel takes fewer planes per workgroup on small grids, and the three momentum solves
share their launches.  A field that repeats a small box over a large one has the small box's
solution repeated, so one step on the large grid (32 planes per workgroup, the last run of
them ragged) is compared with one on the small grid (2 planes), which tests/test_gpu_fluid.py
holds to the oracle.  Both solve the same modes: 1e-12 of the largest value, the bar the solves
have there.
"""
import numpy as np
import pytest

from suguru_amd import workload as W

pytestmark = pytest.mark.gpu
REP, DT, H = 0.0016, 1e-4, 0.25


@pytest.mark.parametrize("ri,rj,kt", [(32, 16, 40), (16, 4, 33)])
def test_repeated_box_keeps_its_solution(ri, rj, kt):
    import torch

    from suguru_amd.fluid import FlowSolver

    small, big = (32, 16, kt), (32 * ri, 16 * rj, kt)
    print(f"case: flow step {big} against {small}", flush=True)
    rng = np.random.default_rng(ri)
    dev = lambda a: torch.from_numpy(a).to("cuda:0")
    inner = [rng.standard_normal((kt, small[1], small[0])) for _ in range(10)]
    got = []
    for shape, rep in ((small, (1, 1, 1)), (big, (1, rj, ri))):
        g = W.make_grid(*shape, H)
        s = FlowSolver(g, REP, DT)
        f = []
        for a in inner:
            b = torch.zeros((kt + 2, shape[1] + 2, shape[0] + 2), dtype=torch.float64, device="cuda:0")
            b[1:-1, 1:-1, 1:-1] = dev(np.tile(a, rep))
            f.append(b.view(-1))
        uo, uoo, p, F = f[:3], f[3:6], f[6], f[7:10]
        un = [torch.zeros_like(p) for _ in range(3)]
        q = torch.zeros_like(p)
        torch.cuda.synchronize()
        s.bounduvw(*uo)
        s.bounduvw(*uoo)
        s.boundp(p)
        s.step(*un, p, q, *uo, *uoo, *F)
        s.sync()
        got.append([a.view(kt + 2, shape[1] + 2, shape[0] + 2) for a in (*un, p, q)])
        s.close()
    for a, b, nm in zip(*got, ("u", "v", "w", "pnew", "p")):
        want = a[:, 1:-1, 1:-1].repeat(1, rj, ri)
        d = (b[:, 1:-1, 1:-1] - want).abs().max()
        assert float(d) <= 1e-12 * float(want.abs().max()), nm
        # the halos are copies of the interior
        assert torch.equal(b[:, :, 0], b[:, :, -2]) and torch.equal(b[:, 0], b[:, -2]), nm
