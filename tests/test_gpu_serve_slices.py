"""Served requests of more paths than a launch takes, rendered a slice of
their passes at a time in turn with others: bit for bit what a plain launch
gives."""
import numpy as np
import pytest

from util import GpuTarget, book_lookat, box_lookat, gpu_params, sha
from venusaur_amd import api

pytestmark = pytest.mark.gpu


# the smallest queue gives launches of 8M paths: three slices of a float image
# and of a double one, slices whose last shares its launch with small
# requests, an image of one pass above a launch, and progressive frames
@pytest.mark.parametrize("kind", ["book", "mem"])
def test_sliced_requests_equal_plain_launches(ctx, book, kind):
    print(f"case: served slices {kind}", flush=True)
    (s, m), look = (book, book_lookat) if kind == "book" else (api.box_scene(3000, 9), box_lookat)
    other = api.Scene(ctx, *api.box_scene(700, 3))
    sc = api.Scene(ctx, s, m)
    jobs = []
    for w, h, spp, fp64, scene in [(1021, 763, 24, False, sc), (128, 130, 1100, True, sc), (64, 36, 2, False, sc),
                                   (4099, 2301, 2, False, sc), (640, 360, 37, False, other), (33, 17, 1, False, other),
                                   (256, 256, 300, False, sc)]:
        t = GpuTarget(w, h, fp64=fp64)
        p = t.bind(gpu_params(w, h, spp, 6, look(w, h), flags=api.ACCUM_FP64 if fp64 else 0))
        jobs.append((scene, p, t))
    frames = (1, 2)
    want, segs = [], []
    for f in frames:
        for scene, p, t in jobs:
            p.subframe_index = f
            segs.append(scene.launch(p).segments)
            want.append((sha(t.accum_host()), sha(t.image_host())))
    for _, _, t in jobs:
        t.accum.zero()
        t.image.zero()
    srv = api.Server(ctx, 4 << 30, tuning=api.Tuning(queue_capacity=1))
    k = 0
    for f in frames:
        ids = []
        for scene, p, t in jobs:
            p.subframe_index = f
            ids.append(srv.submit(scene, p))
        srv.drain()
        for i, (_, p, t) in zip(ids, jobs):
            r = srv.poll(i)
            what = (f, p.width, p.height, p.samples_per_pixel)
            assert r.status == 0 and r.segments == segs[k], what
            assert (sha(t.accum_host()), sha(t.image_host())) == want[k], what
            k += 1
    srv.close()
    sc.close()
    other.close()


# budgets of one footprint and of a little more: slots that shrink and grow
# between a request of several slices and small ones
@pytest.mark.parametrize("factor", [1.0, 1.4, 2.5])
def test_tight_budget_same_results(ctx, book, factor):
    print(f"case: served within a budget of {factor} footprints", flush=True)
    sc = api.Scene(ctx, *book)
    jobs, want = [], []
    for w, h, spp in [(640, 480, 40), (61, 33, 4), (512, 512, 20), (640, 480, 40), (900, 301, 33)]:
        t = GpuTarget(w, h)
        p = t.bind(gpu_params(w, h, spp, 5, book_lookat(w, h)))
        sc.launch(p)
        want.append(sha(t.accum_host()))
        t.accum.zero()
        jobs.append((p, t))
    srv = api.Server(ctx, int(factor * max(api.footprint(p) for p, _ in jobs)), tuning=api.Tuning(queue_capacity=1))
    ids = [srv.submit(sc, p) for p, _ in jobs]
    srv.drain()
    assert [srv.poll(i).status for i in ids] == [0] * len(ids)
    assert [sha(t.accum_host()) for _, t in jobs] == want
    srv.close()
    sc.close()


# the smallest memory a tuning gives a batch is 16M paths: groups of several
# items and of one, an item that fills it exactly, items above it (in double and
# float, several chunks each), counted and not
@pytest.mark.parametrize("count", [False, True])
def test_batch_groups_and_large_items(ctx, book, count):
    print(f"case: batch groups and large items, visits counted: {count}", flush=True)
    scenes = [api.Scene(ctx, *book), api.Scene(ctx, *api.box_scene(3000, 9))]
    jobs, want, segs = [], [], 0
    for i, (w, h, spp, fp64) in enumerate([(512, 512, 40, False), (64, 36, 2, False), (512, 512, 24, False),
                                           (512, 512, 64, False), (640, 480, 70, True), (33, 17, 3, False),
                                           (1024, 768, 33, False), (256, 256, 8, False)]):
        t = GpuTarget(w, h, fp64=fp64)
        flags = (api.ACCUM_FP64 if fp64 else 0) | (api.COUNT_VISITS if count else 0)
        p = t.bind(gpu_params(w, h, spp, 4, (book_lookat, box_lookat)[i % 2](w, h), flags=flags))
        segs += scenes[i % 2].launch(p).segments
        want.append(sha(t.accum_host()))
        t.accum.zero()
        jobs.append((scenes[i % 2], p, t))
    st = api.batch_launch(ctx, [(sc, p) for sc, p, _ in jobs], tuning=api.Tuning(queue_capacity=1))
    assert st.segments == segs and (st.node_visits > 0) == count
    # the first two, the third (5120 paths too many for it), the one of exactly
    # 16M, the last two; and the images of 21.5M and 26M paths in two chunks each
    assert st.iterations == 4 + 2 + 2, st.iterations
    assert [sha(t.accum_host()) for _, _, t in jobs] == want
    for sc in scenes:
        sc.close()
