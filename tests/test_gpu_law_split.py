"""GPU: the membrane law across its splits of the work.

A few capsules are cut into runs of rings over many workgroups, many capsules are one run each
and go in batches of the plan's slots (2048), the selective form packs the selected capsules
first.  No sum depends on the split, so every capsule of a larger batch has the bits it has in a
batch of five; the five are compared with the CPU oracle (tests/test_gpu_membrane.py's bar,
1e-10 of the largest traction component), as is the ordered form.
"""
import ctypes

import numpy as np
import pytest

import _oracle as O
from test_gpu_membrane import D, capsules, oracle_lib

pytestmark = pytest.mark.gpu
GS = 6250.0


def run(torch, plan, xyz, eb, sel=None, ordered=False):
    n = xyz[0].numel()
    out = [torch.full((n,), -7.0, dtype=torch.float64, device="cuda:0") for _ in range(7)]
    torch.cuda.synchronize()
    if sel is not None:
        plan.traction_select_dev(sel, *xyz, GS, eb, *out)
    elif ordered:
        plan.traction_ordered_dev(*xyz, GS, eb, *out)
    else:
        plan.traction_dev(*xyz, GS, eb, *out)
    plan.sync()
    return torch.stack(out).view(7, -1, plan.npts)


@pytest.mark.parametrize("L,eb", [(16, 0.3), (16, 0.0), (2, 0.3), (5, 0.0), (23, 0.3)])
def test_splits_keep_the_bits(L, eb):
    import torch

    from suguru_amd.membrane import MembranePlan

    plan = MembranePlan(L)
    n = plan.npts
    five = [torch.from_numpy(a).to("cuda:0") for a in capsules(L, 5, seed=3 * L + 1)]
    print(f"case: law splits L={L} eb={eb}, 5 capsules", flush=True)
    base = run(torch, plan, five, eb * GS)
    o = oracle_lib()
    for form in (base, run(torch, plan, five, eb * GS, ordered=True)):
        got = form.cpu().numpy()
        for c in range(5):
            want = [np.zeros(n) for _ in range(7)]
            p = [np.ascontiguousarray(a[c * n:(c + 1) * n].cpu().numpy()) for a in five]
            o.mem_traction(L, GS, eb * GS, *[a.ctypes.data_as(D) for a in p],
                           *[w.ctypes.data_as(D) for w in want])
            fmax = max(np.abs(want[k]).max() for k in range(3))
            for k in range(7):
                assert np.abs(got[k, c] - want[k]).max() < (1e-10 * fmax if k < 3 else 1e-12 * max(
                    1.0, np.abs(want[k]).max())), (c, k)
    # 1: every ring its own workgroup; 31, 300: runs of several rings; 1100: one run each, more
    # than the workgroups in flight; 2051: a second batch of three capsules
    for ncap in (1, 31, 300, 1100, 2051):
        print(f"case: law splits L={L} eb={eb}, {ncap} capsules", flush=True)
        idx = torch.arange(ncap, device="cuda:0") % 5
        many = [a.view(5, n)[idx].reshape(-1).contiguous() for a in five]
        got = run(torch, plan, many, eb * GS)
        assert torch.equal(got, base[:, idx]), ncap
        # selected: none, a few (the last one among them), all
        for keep in (torch.zeros(ncap, dtype=torch.bool), torch.arange(ncap) % 97 == (ncap - 1) % 97,
                     torch.ones(ncap, dtype=torch.bool)):
            sel = keep.to(torch.int32).to("cuda:0")
            part = run(torch, plan, many, eb * GS, sel)
            k = keep.to("cuda:0")
            assert torch.equal(part[:, k], base[:, idx[k]]), (ncap, int(keep.sum()))
            assert bool((part[:, ~k] == -7.0).all())
    plan.close()
