"""GPU: the solves at each line length the transforms have a kernel for, and at the lengths beside
them that go through the general one, against numpy's transforms and an elimination in
64 bits.

Tolerance: the one the solves have in tests/test_gpu_fluid.py, 1e-12 of the largest value
(transforms of at most 4096 values round by 1e-14).
"""
import numpy as np
import pytest

import _oracle as O
from suguru_amd import workload as W

pytestmark = pytest.mark.gpu
REP, DT = 0.0016, 1e-4
TOL = 1e-12

# itot 16 .. 2048 and jtot 8 .. 1024 in registers; 4, 8 and 4096 / 4 and 2048 beside them; plane
# counts that leave the last workgroup ragged
SHAPES = [(16, 8, 3), (16, 4, 5), (8, 8, 5), (4, 1024, 3), (32, 1024, 3), (64, 512, 3), (128, 256, 3),
          (256, 128, 5), (512, 64, 3), (1024, 32, 3), (2048, 16, 3), (4096, 8, 2), (16, 2048, 3)]


def solve(g, p):
    """The interior (i, j, k) of solver1d(ne = 2)."""
    a, b, c, _ = O.initsolver(W.make_grid(4, 4, g.ktot, 1 / g.dxi), REP, DT, 2)
    eig = lambda n: -4 * g.dxi**2 * np.sin(np.pi * np.arange(n) / n) ** 2
    xy = eig(g.itot)[:, None] + eig(g.jtot)[None, :]
    f = np.fft.fft2(p, axes=(0, 1))
    d, prev = np.zeros_like(xy), np.zeros_like(f[:, :, 0])
    ds = []
    for k in range(g.ktot):
        z = 1.0 / (b[k] + xy - a[k] * d)
        prev = f[:, :, k] = (f[:, :, k] - a[k] * prev) * z
        d = c[k] * z
        ds.append(d)
    for k in range(g.ktot - 2, -1, -1):
        f[:, :, k] -= ds[k] * f[:, :, k + 1]
    return np.fft.ifft2(f, axes=(0, 1)).real


@pytest.mark.parametrize("shape", SHAPES)
def test_line_lengths_match_oracle(shape):
    import torch

    from suguru_amd.fluid import FlowSolver

    print(f"case: solver1d and step grid {shape}", flush=True)
    g = W.make_grid(*shape, 0.1)
    s = FlowSolver(g, REP, DT)
    rng = np.random.default_rng(shape[0] + shape[1])
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a.reshape(-1, order="F"))).to("cuda:0")
    p = np.asfortranarray(rng.standard_normal(g.shape_f))
    inner = (slice(1, -1),) * 3
    want = solve(g, p[inner])
    t = dev(p)
    torch.cuda.synchronize()
    s.solver1d(t, 2)
    s.sync()
    got = t.cpu().numpy().reshape(g.shape_f, order="F")
    assert np.abs(got[inner] - want).max() <= TOL * np.abs(want).max()
    keep = np.ones(g.shape_f, bool)
    keep[inner] = False
    assert np.array_equal(got[keep].view(np.uint64), p[keep].view(np.uint64))

    # the step's pressure (divergence taken while the x lines are loaded) is fillps and solver1d
    f = [dev(rng.standard_normal(g.shape_f)) for _ in range(10)]
    u, v = ([torch.zeros_like(t) for _ in range(3)] for _ in range(2))
    q, r = torch.zeros_like(t), torch.zeros_like(t)
    torch.cuda.synchronize()
    s.fftuvw(*u, *f)
    s.bounduvw(*u)
    s.fillps(*u, q)
    s.solver1d(q, 1)
    s.step(*v, f[6], r, *f[:6], *f[7:])
    s.sync()
    box = lambda a: a.view(*reversed(g.shape_f))[1:-1, 1:-1, 1:-1]
    assert torch.equal(box(q), box(r))
    s.close()
