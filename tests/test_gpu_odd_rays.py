"""Rays whose roots overflow or are not numbers: the closest hit then depends
on the order in which spheres are tested, and every entry point keeps the one
order (the traversal that counts visits, which the oracle follows)."""
import numpy as np
import pytest

import oracle as O
from venusaur_amd import api
from venusaur_amd.hipmem import DeviceBuffer

pytestmark = pytest.mark.gpu
N = 6000


def _scene(kind, book):
    if kind == "book":
        return book
    if kind == "one":
        return tuple(a[1:].copy() for a in api.box_scene(1, 4))
    if kind == "far":  # centres whose distances overflow when squared
        s, m = api.box_scene(2000, 9)
        s = s.copy()
        for f in ("cx", "cy", "cz", "r"):
            s[f] *= np.float32(1e17)
        return s, m
    return api.box_scene({"lds": 500, "mem": 3000}[kind], 9)


def _rays(s, rng):
    r = np.zeros(N, api.RAY_DT)
    pick = s[rng.integers(0, len(s), N)]
    for f, c in (("ox", "cx"), ("oy", "cy"), ("oz", "cz")):
        r[f] = rng.uniform(-30, 30, N)
        r["d" + f[1]] = pick[c] - r[f] + rng.normal(0, 0.3, N)
    r["tmin"], r["tmax"] = 0.001, 1e16
    return r


def _grow(r, names, by):
    for f in names:
        r[f] = (r[f].astype(np.float64) * by).astype(np.float32)
    r["tmin"], r["tmax"] = 0.0, 3e38


ODD = [("tmax", np.nan), ("tmin", np.nan), ("ox", np.nan), ("dx", np.nan), ("dz", np.nan), ("ox", np.inf),
       ("dy", -np.inf), ("dirs", 1e10), ("dirs", 1e15), ("dirs", 1e18), ("dirs", 1e19), ("dirs", 1e30),
       ("dirs", 1e-25), ("origins", 1e5), ("origins", 1e12), ("origins", 1e19), ("none", 0.0)]


@pytest.mark.parametrize("kind", ["book", "one", "lds", "mem", "far"])
def test_hits_keep_their_order(ctx, book, kind):
    s, m = _scene(kind, book)
    sc = api.Scene(ctx, s, m)
    ob = O.BVH(s)
    rng = np.random.default_rng(5)
    for what, v in ODD:
        print(f"case: odd rays {kind} {what} {v}", flush=True)
        r = _rays(s, rng)
        if what == "dirs":
            _grow(r, ("dx", "dy", "dz"), v)
        elif what == "origins":
            _grow(r, ("ox", "oy", "oz"), v)
        elif what != "none":
            r[what][rng.random(N) < 0.5] = v  # among ordinary ones
        rb = DeviceBuffer.from_array(r)
        got = []
        for trace, stats in ((sc.trace, False), (sc.trace_noalloc, False), (sc.trace, True)):
            h = DeviceBuffer(N * 8)
            h.zero()
            trace(rb.value, N, h.value, stats=stats)
            got.append(h.download(api.HIT_DT))
        want = ob.trace(r)[0]
        for g in got:
            same_t = (g["t"].view(np.uint32) == want["t"].view(np.uint32)) | (np.isnan(g["t"]) & np.isnan(want["t"]))
            assert same_t.all() and (g["prim"] == want["prim"]).all(), (what, v)
    sc.close()
