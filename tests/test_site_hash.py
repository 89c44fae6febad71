"""The site hash's home index (layout.h) over the shapes a scaffold takes: how many
entries a lookup reads on the engine's table, which is the smallest power of two
with two entries per domain slot."""
import ctypes as C
import random

import pytest

from test_engine_host_parity import HOST_LIB, sampler_cls  # noqa: F401


def walk(n, seed):
    r = random.Random(seed)
    p, seen = (0, 0, 0), {(0, 0, 0): None}
    while len(seen) < n:
        q = list(p)
        q[r.randrange(3)] += r.choice((-1, 1))
        p = tuple(q)
        seen[p] = None
    return list(seen)


SHAPES = {
    "sheet_xy": [(x, y, 0) for x in range(8) for y in range(8)],
    "sheet_xz": [(x, 0, z) for x in range(8) for z in range(8)],
    "sheet_yz": [(0, y, z) for y in range(8) for z in range(8)],
    "sheet_far_out": [(x + 1000, y - 500000, 7) for x in range(8) for y in range(8)],
    "sheet_ragged": [(x, y, 0) for x in range(5) for y in range(7)],
    "block": [(x, y, z) for x in range(5) for y in range(5) for z in range(8)],
    "line_x": [(i, 0, 0) for i in range(200)],
    "line_y": [(0, i, 0) for i in range(200)],
    "line_z": [(0, 0, i) for i in range(200)],
    "walk_64": walk(64, 1),
    "walk_200": walk(200, 2),
}


@pytest.mark.parametrize("name", sorted(SHAPES))
def test_lookups_read_few_entries(sampler_cls, name):  # noqa: F811
    home = C.CDLL(HOST_LIB).eh_site_home
    sites = SHAPES[name]
    bits = 6
    while (1 << bits) < 8 * len(sites):
        bits += 1
    n = 1 << bits
    table = [None] * n
    for p in sites:
        i = home(*p, bits)
        assert 0 <= i < n
        while table[i] is not None:
            i = (i + 1) % n
        table[i] = p
    around = {tuple(c + (s if k == a else 0) for k, c in enumerate(p))
              for p in sites for a in range(3) for s in (-1, 1)} - set(sites)

    def entries_read(p):
        i = home(*p, bits)
        for k in range(1, n + 1):
            if table[i] is None or table[i] == p:
                return k
            i = (i + 1) % n

    # a uniform hash reads (1 + 1 / (1 - a)^2) / 2 = 1.15 entries for an empty
    # site at load a = 1/8 (Knuth, TAOCP 6.4), and fewer for an occupied one;
    # half an entry more is left to the shapes' regularity
    for group in (sites, around):
        assert sum(map(entries_read, group)) / len(group) <= 1.65
