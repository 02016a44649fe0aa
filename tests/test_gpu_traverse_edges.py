"""Closest hits of small scenes at the edges of the traversal staged in LDS:
more stacked children than it holds in LDS, and boxes met exactly at their
planes, at the ends of the ray interval and far from the origin."""
import numpy as np
import pytest

import oracle as O
from util import GpuTarget, box_lookat, gpu_params, oracle_params
from venusaur_amd import api
from venusaur_amd.hipmem import DeviceBuffer

pytestmark = pytest.mark.gpu
LDS_NODES, LDS_SPHERES = 256, 769  # what is staged (vz_traverse_lds.h)


def _hits(sc, rays):
    rb, h = DeviceBuffer.from_array(rays), DeviceBuffer(len(rays) * 8)
    sc.trace(rb.value, len(rays), h.value)
    return h.download(api.HIT_DT)


# rays among spheres that all overlap enter nearly every box; either side of
# the tree size that is staged
@pytest.mark.parametrize("n,lds", [(300, True), (500, True), (560, False), (769, False), (770, False)])
def test_overlapping_boxes(ctx, n, lds):
    print(f"case: overlapping boxes n={n}", flush=True)
    rng = np.random.default_rng(n)
    s, m = api.box_scene(n - 1, 5)
    s = s.copy()
    for f in ("cx", "cy", "cz"):
        s[f] = rng.normal(0, 0.5, n).astype(np.float32)
    s["r"] = rng.uniform(1.0, 4.0, n).astype(np.float32)
    rays = np.zeros(4000, api.RAY_DT)
    for f in ("ox", "oy", "oz"):
        rays[f] = rng.uniform(-6, 6, len(rays))
        rays["d" + f[1]] = rng.normal(0, 1, len(rays))
    rays["tmin"], rays["tmax"] = 0.001, 1e16
    rays["tmin"][::7] = -20.0
    sc = api.Scene(ctx, s, m)
    assert (sc.info().num_wide_nodes <= LDS_NODES and n <= LDS_SPHERES) == lds, sc.info().num_wide_nodes
    assert _hits(sc, rays).tobytes() == O.trace_brute(s, rays).tobytes()
    t = GpuTarget(40, 30)
    sc.launch(t.bind(gpu_params(40, 30, 3, 12, box_lookat(40, 30))))
    want, _, _ = O.render(s, m, oracle_params(40, 30, 3, 12, box_lookat(40, 30)), bvh=O.BVH(s))
    assert np.array_equal(t.accum_host(), want)
    sc.close()


@pytest.mark.parametrize("n,lds", [(400, True), (900, False)])
@pytest.mark.parametrize("away", [0.0, 1e4, 1e6])
def test_planes_and_interval_ends(ctx, n, lds, away):
    print(f"case: planes and interval ends n={n} away={away}", flush=True)
    rng = np.random.default_rng([n, int(away)])
    s, m = api.box_scene(n, 9)
    s, m = s[1:].copy(), m[1:].copy()  # without the ground
    s["r"] = rng.uniform(0.5, 3.0, n).astype(np.float32)
    for f, k in (("cx", 1.0), ("cy", -0.7), ("cz", 0.4)):
        s[f] += np.float32(k * away)
    sc = api.Scene(ctx, s, m)
    assert (sc.info().num_wide_nodes <= LDS_NODES) == lds, sc.info().num_wide_nodes
    count = 3000
    rays = np.zeros(count, api.RAY_DT)
    pick = s[rng.integers(0, n, count)]
    cen = np.stack([pick["cx"], pick["cy"], pick["cz"]], 1)
    axis = rng.integers(0, 3, count)
    d = rng.normal(0, 1, (count, 3)).astype(np.float32)
    along = rng.random(count) < 0.5  # down an axis, at the sphere's own planes
    d[along] = 0.0
    d[np.arange(count)[along], axis[along]] = rng.choice([-1.0, 1.0], along.sum())
    o = cen - d * rng.uniform(5, 50, count).astype(np.float32)[:, None]
    side = (axis + 1) % 3
    o[np.arange(count)[along], side[along]] += (pick["r"] * rng.choice([-1.0, 0.0, 1.0], count).astype(np.float32))[along]
    for k, f in enumerate("xyz"):
        rays["o" + f], rays["d" + f] = o[:, k], d[:, k]
    rays["tmin"], rays["tmax"] = 0.001, 1e16
    first = O.trace_brute(s, rays)
    assert _hits(sc, rays).tobytes() == first.tobytes()
    hit = first["prim"] != api.MISS
    assert hit.sum() > count // 3
    for end in (first["t"], np.nextafter(first["t"], np.float32(0)), np.nextafter(first["t"], np.float32(np.inf))):
        r = rays[hit].copy()
        r["tmax"] = end[hit]
        assert _hits(sc, r).tobytes() == O.trace_brute(s, r).tobytes()
        r = rays[hit].copy()
        r["tmin"] = end[hit]
        assert _hits(sc, r).tobytes() == O.trace_brute(s, r).tobytes()
    sc.close()


# either side of the size from which many workgroups refit the nodes across
# workgroups' ranges, and of the one it was before
@pytest.mark.parametrize("n", [393216, 393217, 655360, 655361])
def test_refit_lines(ctx, n):
    print(f"case: refit of {n} spheres", flush=True)
    s, m = api.box_scene(n - 1, 7)
    sc = api.Scene(ctx, s, m)
    s["cx"][1:] += np.random.default_rng(n).uniform(-0.2, 0.2, n - 1).astype(np.float32)
    sc.update_spheres(s)
    rays = np.zeros(400, api.RAY_DT)
    rng = np.random.default_rng([n, 1])
    pick = s[rng.integers(0, n, len(rays))]
    for f, c in (("ox", "cx"), ("oy", "cy"), ("oz", "cz")):
        rays[f] = rng.uniform(-100, 100, len(rays))
        rays["d" + f[1]] = pick[c] - rays[f]
    rays["tmin"], rays["tmax"] = 0.001, 1e16
    assert _hits(sc, rays).tobytes() == O.trace_brute(s, rays).tobytes()
    sc.close()


# without stats the call only enqueues: captured once, replayed on other rays,
# scenes in LDS and in memory, odd rays (a NaN limit) among them
@pytest.mark.parametrize("kind", ["lds", "mem"])
def test_captured_trace(ctx, book, kind):
    print(f"case: captured hits {kind}", flush=True)
    torch = pytest.importorskip("torch")
    s, m = book if kind == "lds" else api.box_scene(5000, 9)
    sc = api.Scene(ctx, s, m)
    n = 30001

    def make(seed):
        rng = np.random.default_rng(seed)
        r = np.zeros(n, api.RAY_DT)
        pick = s[rng.integers(0, len(s), n)]
        for f, c in (("ox", "cx"), ("oy", "cy"), ("oz", "cz")):
            r[f] = rng.uniform(-30, 30, n)
            r["d" + f[1]] = pick[c] - r[f]
        r["tmin"], r["tmax"] = 0.001, 1e16
        r["tmax"][::97] = np.nan
        return r

    dev = lambda a: torch.from_numpy(a.view(np.uint8).reshape(-1).copy()).cuda()  # noqa: E731
    rays, hits = dev(make(0)), torch.zeros(n * 2, dtype=torch.int32, device="cuda")
    api.check(api.lib().vzTraceClosestNoAlloc(sc.h, rays.data_ptr(), n, hits.data_ptr(), None, None))
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        st = torch.cuda.current_stream().cuda_stream
        api.check(api.lib().vzTraceClosestNoAlloc(sc.h, rays.data_ptr(), n, hits.data_ptr(), st, None))
    for seed in range(1, 5):
        r = make(seed)
        rays.copy_(dev(r))
        hits.zero_()
        g.replay()
        torch.cuda.synchronize()
        got = hits.cpu().numpy().view(np.uint8).view(api.HIT_DT)
        want = O.BVH(s).trace(r)[0]
        same_t = (got["t"].view(np.uint32) == want["t"].view(np.uint32)) | (np.isnan(got["t"]) & np.isnan(want["t"]))
        assert same_t.all() and (got["prim"] == want["prim"]).all(), seed
        sc2 = api.Scene(ctx, s[:100].copy(), m[:100].copy())  # eager work of the program between replays
        sc2.close()
    sc.close()
