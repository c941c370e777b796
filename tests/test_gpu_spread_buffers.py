"""GPU: the spread's work buffers by capsule count.  A call with fewer capsules than an earlier one
on the same context allocates nothing, so that a graph captured of the earlier call stays valid; a
capsule whose few points lie far apart (far more items than its points suggest) spreads to the
oracle's bits.
"""
import numpy as np
import pytest

import _oracle as O
from suguru_amd import IBTransfer, workload as W

pytestmark = pytest.mark.gpu


def dev(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def spread(t, g, caps, f, n):
    """The spread of the first n capsules."""
    import torch

    m = int(caps.cap_off[n])
    args = [dev(caps.cap_off[:n + 1]), *[dev(a[:m]) for a in (caps.x, caps.y, caps.z, *f, caps.area)]]
    out = [torch.full((g.ncells_halo,), np.nan, dtype=torch.float64, device="cuda:0")
           for _ in range(3)]
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    t.spread_dev(*args, *out)
    t.sync()
    return out, free - torch.cuda.mem_get_info()[0]


def test_fewer_capsules_allocate_nothing():
    g = W.make_grid(128, 100, 90)
    rng = np.random.default_rng(11)
    n, r = 30, 10.6
    cen = rng.uniform(0.0, 1.0, (n, 3)) * [g.lx, g.ly, g.lz - 2 * r * g.dx]
    cen[:, 2] += r * g.dx
    caps = W.build_capsules(cen, np.full(n, r * g.dx), [16] * n)
    f = W.forces(caps.npts, 1)
    t = IBTransfer(g, 0)
    try:
        spread(t, g, caps, f, n)
        for k in (20, 12, 4, 1, n):
            print(f"case: spread of {k} capsules after {n}", flush=True)
            assert spread(t, g, caps, f, k)[1] == 0
    finally:
        t.close()


def test_few_points_far_apart():
    print("case: spread of one capsule of 98 points all over the grid", flush=True)
    g = W.make_grid(128, 100, 90)
    rng = np.random.default_rng(12)
    caps = W.build_capsules(np.array([[0.5 * g.lx, 0.5 * g.ly, 0.5 * g.lz]]), np.full(1, g.dx), [6])
    for a, l in ((caps.x, g.lx), (caps.y, g.ly), (caps.z, g.lz)):
        a[:] = rng.uniform(0.0, l, caps.npts)
    f = W.forces(caps.npts, 2)
    t = IBTransfer(g, 0)
    try:
        out, _ = spread(t, g, caps, f, 1)
        want = O.lagr2eulr(g, caps.cap_off, caps.x, caps.y, caps.z, *f, caps.area)
        for a, b in zip(out, want):
            assert np.array_equal(a.cpu().numpy().view(np.uint64),
                                  b.reshape(-1, order="F").view(np.uint64))
    finally:
        t.close()
