"""Plain launches (vzLaunch, the persistent path kernels) at the edges of
their tiles, units and chunks, bit for bit against the CPU oracle; a frame of
more passes than one chunk holds against the megakernel."""
import sys

import numpy as np
import pytest

import oracle as O
from util import GpuTarget, book_lookat, box_lookat, gpu_params, oracle_params
from venusaur_amd import api
from venusaur_amd.hipmem import DeviceBuffer

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _scene(kind, book):
    if kind == "book":
        return book, book_lookat
    if kind == "one":  # a single sphere: no tree
        s, m = api.box_scene(1, 4)
        return (s[1:].copy(), m[1:].copy()), box_lookat
    n = {"lds": 500, "mem": 700}[kind]  # either side of the tree size staged in LDS
    return api.box_scene(n, 9), box_lookat


# smaller than a tile, exactly one, one pixel more, each tile shape, odd
# sizes; passes below, at and above a unit's 8, and not a multiple of it
@pytest.mark.parametrize("kind,w,h,spp,depth", [
    ("book", 2, 2, 1, 50), ("book", 7, 3, 9, 8), ("book", 3, 41, 2, 4), ("book", 8, 8, 8, 50),
    ("book", 9, 7, 17, 3), ("book", 65, 33, 3, 1), ("book", 131, 67, 5, 50), ("one", 16, 9, 3, 6),
    ("lds", 33, 17, 7, 16), ("mem", 33, 17, 7, 16), ("mem", 2, 64, 12, 255)])
@pytest.mark.parametrize("fp64", [False, True])
def test_launch_edges(ctx, book, kind, w, h, spp, depth, fp64):
    say(f"case: plain launch {kind} {w}x{h} spp={spp} depth={depth} fp64={fp64}")
    (s, m), look = _scene(kind, book)
    cam = look(w, h)
    sc = api.Scene(ctx, s, m)
    tgt = GpuTarget(w, h, fp64=fp64)
    ob = O.BVH(s)
    want = None
    for frame in (1, 2):
        p = gpu_params(w, h, spp, depth, cam, subframe=frame, flags=api.ACCUM_FP64 if fp64 else 0)
        st = sc.launch(tgt.bind(p))
        want, img, ost = O.render(s, m, oracle_params(w, h, spp, depth, cam, subframe=frame, accum_fp64=fp64), bvh=ob,
                                  accum=want)
        assert np.array_equal(tgt.accum_host(), want), frame
        assert np.abs(tgt.image_host().astype(int) - img.astype(int)).max() <= 1
        assert (st.segments, st.hits, st.paths) == (ost.segments, ost.hits, w * h * spp)
    p.flags |= api.COUNT_VISITS
    p.subframe_index = 1
    st = sc.launch(p)
    _, _, ost = O.render(s, m, oracle_params(w, h, spp, depth, cam), bvh=ob)
    assert (st.segments, st.node_visits, st.sphere_tests) == (ost.segments, ost.node_visits, ost.sphere_tests)
    sc.close()


@pytest.mark.parametrize("fp64", [False, True])
def test_launch_of_several_chunks(ctx, book, fp64):
    """2048x2048 holds 64 passes in a chunk: 131 passes are three chunks whose
    sums and camera seeds carry over, the last one shorter."""
    say(f"case: plain launch of several chunks fp64={fp64}")
    s, m = book
    sc = api.Scene(ctx, s, m)
    out = []
    flags = api.ACCUM_FP64 if fp64 else 0
    for extra in (0, api.MEGAKERNEL):
        tgt = GpuTarget(2048, 2048, fp64=fp64)
        st = sc.launch(tgt.bind(gpu_params(2048, 2048, 131, 2, book_lookat(2048, 2048), flags=flags | extra)))
        out.append((st.segments, st.paths, tgt.accum_host(), tgt.image_host()))
    assert out[0][:2] == out[1][:2]
    assert np.array_equal(out[0][2], out[1][2]) and np.array_equal(out[0][3], out[1][3])
    sc.close()


# without stats the rays go through persistent waves (a small scene in LDS):
# sizes around a wave, a workgroup and all resident waves, and ray intervals
# that start behind the origin, end before it, or are empty
@pytest.mark.parametrize("kind", ["book", "one", "lds", "mem"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 769, 49153, 500001])
def test_trace_without_stats(ctx, book, kind, n):
    say(f"case: hits without stats {kind} n={n}")
    (s, m), look = _scene(kind, book)
    rng = np.random.default_rng([n, 3])
    rays = np.zeros(n, api.RAY_DT)
    pick = s[rng.integers(0, len(s), n)]
    for f, c in (("ox", "cx"), ("oy", "cy"), ("oz", "cz")):
        rays[f] = rng.uniform(-30, 30, n)
        rays["d" + f[1]] = pick[c] - rays[f] + rng.normal(0, 0.3, n)
    rays["dx"][::17] = 0.0
    rays["dy"][::23] = 0.0
    rays["tmin"], rays["tmax"] = 0.001, 1e16
    k = rng.integers(0, 6, n)
    rays["tmin"][k == 1], rays["tmax"][k == 1] = -50.0, 50.0
    rays["tmin"][k == 2], rays["tmax"][k == 2] = -1e16, 1e16
    rays["tmin"][k == 3], rays["tmax"][k == 3] = 0.0, 0.5
    rays["tmin"][k == 4], rays["tmax"][k == 4] = 0.9, 0.2
    sc = api.Scene(ctx, s, m)
    rb = DeviceBuffer.from_array(rays)
    hits = []
    for call in (sc.trace, sc.trace_noalloc):
        h = DeviceBuffer(n * 8)
        call(rb.value, n, h.value)
        hits.append(h.download(api.HIT_DT))
    want = O.trace_brute(s, rays[:20000])
    assert hits[0][:20000].tobytes() == want.tobytes()
    h = DeviceBuffer(n * 8)
    sc.trace(rb.value, n, h.value, stats=True)
    assert hits[0].tobytes() == hits[1].tobytes() == h.download(api.HIT_DT).tobytes()
    sc.close()


# scenes in memory whose rays enter nearly every box: more stacked children
# than the LDS entries of a lane, full leaf queues, ties between copies of a
# sphere; then refitted to other places
@pytest.mark.parametrize("n", [770, 1000, 3001, 20000])
@pytest.mark.parametrize("copies", [1, 3])
def test_trace_overlapping_boxes(ctx, n, copies):
    say(f"case: hits among overlapping boxes n={n} copies={copies}")
    rng = np.random.default_rng([n, copies])
    s, m = api.box_scene(n - 1, 5)
    s, m = s.copy(), m.copy()
    for f in ("cx", "cy", "cz"):
        s[f] = np.tile(rng.normal(0, 0.5, n // copies + 1), copies)[:n].astype(np.float32)
    s["r"] = np.tile(rng.uniform(1.0, 4.0, n // copies + 1), copies)[:n].astype(np.float32)
    rays = np.zeros(4000, api.RAY_DT)
    for f in ("ox", "oy", "oz"):
        rays[f] = rng.uniform(-6, 6, len(rays))
        rays["d" + f[1]] = rng.normal(0, 1, len(rays))
    rays["tmin"], rays["tmax"] = 0.001, 1e16
    rays["tmin"][::7] = -20.0
    sc = api.Scene(ctx, s, m)
    rb = DeviceBuffer.from_array(rays)
    for moved in (False, True):
        if moved:
            s["cx"] += rng.normal(0, 2.0, n).astype(np.float32)
            sc.update_spheres(s)
        out = []
        for stats in (False, True):
            h = DeviceBuffer(len(rays) * 8)
            sc.trace(rb.value, len(rays), h.value, stats=stats)
            out.append(h.download(api.HIT_DT))
        assert out[0].tobytes() == out[1].tobytes() == O.trace_brute(s, rays).tobytes(), moved
    sc.close()


# a tree whose wide levels go on far below its wide ones: beside a box of
# spheres, ever smaller cells of the Morton grid with one sphere each and a
# crowd in the last one
@pytest.mark.parametrize("n", [6000, 30000, 140000])
def test_uneven_tree(ctx, n):
    say(f"case: uneven tree n={n}")
    s, m = api.box_scene(n, 3)
    s, m = s[1:].copy(), m[1:].copy()
    lo = np.array([s[f].min() for f in ("cx", "cy", "cz")])
    ext = float(max(s[f].max() - s[f].min() for f in ("cx", "cy", "cz")))
    chain = [lo + ext * 2.0 ** -k * np.eye(3)[a] for k in range(1, 11) for a in range(3)]
    crowd = lo + np.random.default_rng(n).uniform(0, ext / 2048, (min(n // 3, 4000), 3))
    extra = np.concatenate([chain, crowd])
    keep = np.ones(len(s), bool)  # the box leaves the chain's octant: nothing else there
    for a, f in enumerate(("cx", "cy", "cz")):
        keep &= s[f] < lo[a] + ext * 0.45
    s, m = s[~keep], m[~keep]
    t = np.zeros(len(extra), s.dtype)
    for a, f in enumerate(("cx", "cy", "cz")):
        t[f] = extra[:, a]
    t["r"] = ext * 1e-5
    s = np.concatenate([s, t])
    m = np.concatenate([m, np.resize(m, len(t))])
    sc = api.Scene(ctx, s, m)
    ob = O.BVH(s)
    assert sc.info().num_prims > 2048 and sc.info().wide_depth == ob.wide_depth()
    say(f"wide depth {ob.wide_depth()}")
    assert sc.download_wide().tobytes() == ob.wide_nodes().tobytes()
    rng = np.random.default_rng([n, 1])
    rays = np.zeros(3000, api.RAY_DT)
    pick = s[rng.integers(0, len(s), len(rays))]
    for f, c in (("ox", "cx"), ("oy", "cy"), ("oz", "cz")):
        rays[f] = rng.uniform(lo.min() - ext, lo.min() + 2 * ext, len(rays))
        rays["d" + f[1]] = pick[c] - rays[f]
    rays["tmin"], rays["tmax"] = 0.001, 1e16
    rb = DeviceBuffer.from_array(rays)
    out = []
    for stats in (False, True):
        h = DeviceBuffer(len(rays) * 8)
        sc.trace(rb.value, len(rays), h.value, stats=stats)
        out.append(h.download(api.HIT_DT))
    assert out[0].tobytes() == out[1].tobytes() == O.trace_brute(s, rays).tobytes()
    sc.close()


# launches of few paths, whose tiles' passes are split among waves: from one
# path a wave to whole tiles, plain and in a batch
@pytest.mark.parametrize("kind", ["book", "mem"])
@pytest.mark.parametrize("w,h,spp", [(2, 2, 1), (8, 8, 1), (64, 36, 2), (57, 31, 5), (100, 60, 4), (128, 128, 12),
                                     (160, 160, 13)])
def test_launches_of_few_paths(ctx, book, kind, w, h, spp):
    say(f"case: few paths {kind} {w}x{h} spp={spp}")
    (s, m), look = _scene(kind, book)
    cam = look(w, h)
    sc = api.Scene(ctx, s, m)
    want, _, ost = O.render(s, m, oracle_params(w, h, spp, 12, cam), bvh=O.BVH(s))
    tgt = GpuTarget(w, h)
    st = sc.launch(tgt.bind(gpu_params(w, h, spp, 12, cam)))
    assert np.array_equal(tgt.accum_host(), want) and st.segments == ost.segments
    two = [GpuTarget(w, h), GpuTarget(w, h)]
    st = api.batch_launch(ctx, [(sc, t.bind(gpu_params(w, h, spp, 12, cam))) for t in two])
    assert all(np.array_equal(t.accum_host(), want) for t in two) and st.segments == 2 * ost.segments
    sc.close()
