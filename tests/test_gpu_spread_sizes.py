"""GPU: the spread's item sizes and set-up launches by capsule count, bit for bit against the oracle.

Few capsules get items of 256, 512 or 1024 cells instead of 2048, and up to 1024 capsules have
their item offsets and source lists made inside the item kernel; capsules here touch, cross
the periodic boundaries and reach both walls, so that items have several sources.  The sums run in
the reference's order whatever the items: every bit of the force and normal fields is the
oracle's, through the allocating and the no-allocation entry points.
"""
import numpy as np
import pytest

import _oracle as O
from suguru_amd import IBTransfer, workload as W

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a).reshape(-1).view(np.uint64)


@pytest.mark.parametrize("grid,ncap,radius,degree", [
    ((64, 64, 64), 1, 8.0, 12),       # 256-cell items
    ((45, 38, 33), 3, 6.3, 8),        # the same, odd extents
    ((96, 64, 60), 12, 10.6, 16),     # 512
    ((128, 100, 90), 40, 10.6, 16),   # 1024
    ((128, 100, 90), 300, 4.0, 6),    # 2048, fused set-up
    ((150, 130, 100), 1025, 2.5, 3),  # 2048, separate scan and source launches
])
def test_spread_bits_by_capsule_count(grid, ncap, radius, degree):
    import torch

    print(f"case: spread {grid}, {ncap} capsules of radius {radius}h, degree {degree}", flush=True)
    g = W.make_grid(*grid)
    rng = np.random.default_rng(ncap)
    cen = rng.uniform(0.0, 1.0, (ncap, 3)) * [g.lx, g.ly, g.lz - 2 * radius * g.dx]
    cen[:, 2] += radius * g.dx  # touching the walls at most
    caps = W.build_capsules(cen, np.full(ncap, radius * g.dx), [degree] * ncap)
    f = W.forces(caps.npts, ncap + 1)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    t = IBTransfer(g, 0)
    try:
        off = dev(caps.cap_off)
        p = [dev(a) for a in (caps.x, caps.y, caps.z)]
        d = [dev(a) for a in (*f, caps.area)]
        for kw, fn in ((dict(), O.lagr2eulr), (dict(noalloc=True), O.lagr2eulr),
                       (dict(cc=True), O.lagr2eulrind)):
            out = [torch.full((g.ncells_halo,), np.nan, dtype=torch.float64, device="cuda:0")
                   for _ in range(3)]
            torch.cuda.synchronize()
            t.spread_dev(off, *p, *d, *out, **kw)
            t.sync()
            want = fn(g, caps.cap_off, caps.x, caps.y, caps.z, *f, caps.area)
            for a, b, nm in zip(out, want, "xyz"):
                assert np.array_equal(bits(a.cpu().numpy()), bits(b.reshape(-1, order="F"))), (kw, nm)
    finally:
        t.close()
