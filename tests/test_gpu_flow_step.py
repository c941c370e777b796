"""GPU: fld_step against the sequence of its parts (fftuvw, bounduvw, fillps, solver1d, boundp, correc,
pnew += p, the halos of all), whole arrays with their halos, bit for bit, over the line lengths and
plane shapes that the transforms, the correction and the halo pass index by.
"""
import numpy as np
import pytest

from suguru_amd import workload as W

pytestmark = pytest.mark.gpu
SHAPES = [(4, 4, 2), (4, 64, 3), (8, 8, 5), (16, 8, 3), (4, 1024, 3), (32, 32, 33), (64, 32, 5), (32, 256, 32),
          (256, 32, 7), (128, 64, 31), (128, 128, 6), (1024, 32, 3), (2048, 16, 3), (4096, 8, 2), (16, 2048, 3)]


@pytest.mark.parametrize("shape", SHAPES)
def test_step_is_the_sequence_of_its_parts(shape):
    import torch

    from suguru_amd.fluid import FlowSolver

    print(f"case: step and its parts, grid {shape}", flush=True)
    g = W.make_grid(*shape, 0.1)
    s = FlowSolver(g, 0.0016, 1e-4)
    rng = np.random.default_rng(shape[0] + 3 * shape[1])
    dev = lambda: torch.from_numpy(rng.standard_normal(g.ncells_halo)).to("cuda:0")
    old, pnew, force, new, p = [dev() for _ in range(6)], dev(), [dev() for _ in range(3)], \
        [dev() for _ in range(3)], dev()
    want, wp, wpn = [t.clone() for t in new], p.clone(), pnew.clone()
    torch.cuda.synchronize()
    s.step(*new, pnew, p, *old, *force)

    s.fftuvw(*want, *old, wpn, *force)
    s.bounduvw(*want)
    s.fillps(*want, wp)
    s.solver1d(wp, 1)
    s.boundp(wp)
    s.correc(*want, wp)
    s.bounduvw(*want)
    s.sync()
    inner = lambda t: t.view(g.ktot + 2, g.jtot + 2, g.itot + 2)[1:-1, 1:-1, 1:-1]
    inner(wpn).add_(inner(wp))
    torch.cuda.synchronize()
    s.boundp(wpn)
    s.sync()
    for name, a, b in zip(("u", "v", "w", "p", "pnew"), (*new, p, pnew), (*want, wp, wpn)):
        assert torch.equal(a.view(torch.int64), b.view(torch.int64)), name
    s.close()
