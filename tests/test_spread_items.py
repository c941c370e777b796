"""CPU: the rules of the spread's work items (csrc/obj_items.hpp), compiled for the host: boxes are
cut into items within each limit, the buffers' capacity never falls with the capsule count, and a
launch takes smaller items only where they fit.
"""
import ctypes
import itertools
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "suguru_amd", "csrc")
HOST = """
#include "obj_items.hpp"
using namespace ibx;
extern "C" {
long long capacity(long long n) { return obj_item_capacity(n); }
int choice(const int* tot, int icap) { return obj_choice(tot, icap); }
void limit(int e, int* o) { o[0] = obj_limit(e).bx, o[1] = obj_limit(e).nc; }
void grid(int x, int y, int z, int e, int* o) {
  const int b[6] = {1, x, 1, y, 0, z - 1};
  const ObjGrid g(b, obj_limit(e));
  o[0] = g.cx, o[1] = g.cy, o[2] = g.cz, o[3] = g.nx, o[4] = g.ny, o[5] = g.nz, o[6] = g.count();
}
void packed(const int* c, int* o) {
  o[0] = c[0];
  for (int e = 1; e < OB_LIMITS; ++e) o[e] = obj_unpack(obj_pack(c), e);
}
}
"""


@pytest.fixture(scope="module")
def items(tmp_path_factory):
    d = tmp_path_factory.mktemp("items")
    (d / "host.cpp").write_text(HOST)
    so = str(d / "host.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-I", CSRC,
                    str(d / "host.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)
    lib.capacity.restype = ctypes.c_longlong
    lib.capacity.argtypes = [ctypes.c_longlong]
    return lib


def ints(*v):
    return (ctypes.c_int * len(v))(*v)


def test_capacity_grows_with_the_capsules_alone(items):
    cap = [items.capacity(n) for n in range(3000)]
    assert all(b >= a for a, b in zip(cap, cap[1:]))
    assert all(c >= 64 * n + 1024 for n, c in enumerate(cap))


def test_items_cover_a_box_within_their_limit(items):
    sides = [1, 2, 15, 16, 17, 31, 32, 33, 48, 65, 71, 100]
    o, l = ints(*[0] * 7), ints(0, 0)
    for x, y, z in itertools.product(sides, sides, [1, 2, 5, 16, 31, 33, 70]):
        for e in range(4):
            items.grid(x, y, z, e, o)
            items.limit(e, l)
            cx, cy, cz, nx, ny, nz, n = o
            assert n == cx * cy * cz and max(nx, ny) <= l[0] and nz <= 32 and nx * ny * nz <= l[1]
            for c, s, full in ((cx, nx, x), (cy, ny, y), (cz, nz, z)):
                assert (c - 1) * s < full <= c * s, (x, y, z, e)


def test_small_items_only_where_they_fit(items):
    rng = np.random.default_rng(3)
    for _ in range(2000):
        tot = np.cumsum(rng.integers(1, 600, 4))
        icap = int(rng.integers(1, 2500))
        e, free = (items.choice(ints(*map(int, tot)), c) for c in (icap, 1 << 20))
        fits = [k for k in range(free + 1) if tot[k] <= icap]
        assert e == (max(fits) if fits else 0)


@pytest.mark.parametrize("ncap,limit", [(4, 3), (16, 2), (24, 2), (30, 1), (60, 1), (76, 0), (226, 0)])
def test_size_by_the_items_of_the_boxes(items, ncap, limit):
    """Degree-16 capsules of radius 10.6h, 24 or 25 cells wide with their windows: 8 items of 2048
    cells each, whose 578 points would suggest 3."""
    tot, o = [], ints(*[0] * 7)
    for e in range(4):
        items.grid(25, 24, 24, e, o)
        tot.append(ncap * o[6])
    assert tot[0] == 8 * ncap
    assert items.choice(ints(*tot), items.capacity(ncap)) == limit


def test_counts_survive_the_packing(items):
    o, top = ints(0, 0, 0, 0), 1 << 20  # 256 capsules' saturated counts add up in an int
    for c in [(0, 0, 0, 0), (1, 2, 3, 4), (9, top - 1, top, top + 1), (5, 2**31 - 1, 0, 2**31 - 1)]:
        items.packed(ints(*c), o)
        assert list(o) == [c[0], *(min(v, top) for v in c[1:])]
    assert 256 * top < 2**31
