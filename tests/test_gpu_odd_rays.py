"""Rays whose roots overflow or are not numbers: the closest hit then depends
on the order in which spheres are tested, and every entry point keeps the one
order (the traversal that counts visits, which the oracle follows)."""
import numpy as np
import pytest

import oracle as O
from util import GpuTarget, book_lookat, gpu_params
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
        with np.errstate(over="ignore"):
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


def _odd_launch(what, p, m):
    if what == "far view":
        p.w[:] = [x * 1e19 for x in p.w]
    elif what == "far eye":
        p.origin[:] = [x * 1e18 for x in p.origin]
    elif what == "no frame":
        p.u[:] = [0.0, 0.0, 0.0]
    elif what == "fuzz":
        m["type"][5::7], m["fuzz"][5::7] = api.METAL, np.float32(3e38)
    elif what == "index":
        m["type"][5::7], m["ir"][5::7] = api.DIELECTRIC, np.float32(np.nan)
    elif what == "index 0":
        m["type"][5::7], m["ir"][5::7] = api.DIELECTRIC, np.float32(0.0)


# plain, in a batch with an ordinary item, and served, against the megakernel,
# which walks every ray in the one order
@pytest.mark.parametrize("kind", ["book", "mem", "far"])
@pytest.mark.parametrize("what", ["far view", "far eye", "no frame", "fuzz", "index", "index 0", "none"])
def test_launches_keep_their_order(ctx, book, kind, what):
    print(f"case: odd launch {kind} {what}", flush=True)
    s, m = (a.copy() for a in _scene(kind, book))
    p = gpu_params(96, 54, 4, 8, book_lookat(96, 54))
    _odd_launch(what, p, m)
    sc = api.Scene(ctx, s, m)
    ordinary = api.Scene(ctx, *book)
    q = gpu_params(96, 54, 4, 8, book_lookat(96, 54))
    out = []
    for form in ("mega", "plain", "batch", "serve"):
        t, u = GpuTarget(96, 54), GpuTarget(96, 54)
        p.flags = api.MEGAKERNEL if form == "mega" else 0
        t.bind(p)
        u.bind(q)
        if form in ("mega", "plain"):
            st = sc.launch(p)
            segs = st.segments
            ordinary.launch(q)
            assert form == "mega" or (st.node_visits, st.sphere_tests) == (0, 0)
        elif form == "batch":
            st = api.batch_launch(ctx, [(sc, p), (ordinary, q)])
            assert (st.node_visits, st.sphere_tests) == (0, 0)
            segs = None
        else:
            srv = api.Server(ctx, 1 << 30)
            ids = [srv.submit(sc, p), srv.submit(ordinary, q)]
            srv.drain()
            segs = srv.poll(ids[0]).segments
            srv.close()
        out.append((form, segs, t.accum_host(), u.accum_host()))
    for form, segs, a, b in out[1:]:
        assert np.array_equal(a, out[0][2], equal_nan=True), form
        assert np.array_equal(b, out[0][3], equal_nan=True), form
        assert segs in (None, out[0][1]), form
    sc.close()
    ordinary.close()
