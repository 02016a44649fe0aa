"""What libvz.so does on the host, without a GPU: run in a process of its own
over tests/host_hip, a stand-in for the HIP runtime whose device memory is
host memory and whose kernels do nothing."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, sys
hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
for f in ("host_hip_used", "host_hip_peak", "host_hip_log"):
    getattr(hip, f).restype = C.c_size_t
hip.host_hip_limit.argtypes = [C.c_size_t]
hip.host_hip_launches.argtypes = [C.c_char_p]
FREED = C.CFUNCTYPE(None)
hip.host_hip_on_free.argtypes = [FREED, C.c_size_t]
import time
import numpy as np
from venusaur_amd import api
MB = 1 << 20

def calls():
    buf = C.create_string_buffer(hip.host_hip_log(None, 0) + 1)
    hip.host_hip_log(buf, len(buf))
    return buf.value.decode().split("\\n")[:-1]

def params(w, h, spp, flags=0):
    p = api.launch_params(w, h, spp, 8, [13, 2, 3], [0, 0, 0], 20.0, 0.1, 10.0, flags=flags)
    p.accum = 256  # no kernel runs: never read
    return p

ctx = api.Context(0)
scene = api.Scene(ctx, *api.box_scene(500, 1))
"""


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    out = str(tmp_path_factory.mktemp("host_hip") / "libhost_hip.so")
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(HERE, "host_hip", "host_hip.cpp"), "-o", out], check=True)
    return out


def run(stand_in, code):
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, stand_in, ROOT], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_context_cannot_go_while_a_scene_gives_back_its_memory(stand_in):
    """A scene's block returns to its context's pool: until that is done the
    context counts the scene as alive.  4e6 spheres are above what the pool
    keeps, so their block is freed inside vzSceneDestroy; there, vzDestroy
    (another thread's, say) has to refuse."""
    run(stand_in, """
scene.close()
big = api.Scene(ctx, *api.box_scene(4_000_000, 1))
seen = []
cb = FREED(lambda: seen.append(api.lib().vzDestroy(ctx.h)))
hip.host_hip_on_free(cb, 1 << 30)
assert api.lib().vzSceneDestroy(big.h) == 0
assert seen == [1], seen
hip.host_hip_on_free(FREED(), 0)
assert api.lib().vzDestroy(ctx.h) == 0
ctx.h = big.h = None
""")


def test_little_memory_makes_more_chunks(stand_in):
    """2048x2048 at 131 samples in double takes 44 passes at a time (2.95 GB)
    and 117 MB of sums.  With room for the first alone the launch goes on in
    smaller chunks, for which the larger buffer is given back."""
    run(stand_in, """
p = params(2048, 2048, 131, api.ACCUM_FP64)
base = hip.host_hip_used()
hip.host_hip_limit(base + 2900 * MB)
for _ in range(2):
    st = scene.launch(p)
    assert st.iterations == 6, st.iterations   # 22 passes each
    assert hip.host_hip_used() <= base + 2900 * MB
other = api.Context(0)
s2 = api.Scene(other, *api.box_scene(500, 1))
hip.host_hip_limit(hip.host_hip_used() + 250 * MB)
st = s2.launch(p)
assert st.iterations == 66, st.iterations      # two passes (134 MB) at a time
third = api.Context(0)
hip.host_hip_limit(1 << 60)
s3 = api.Scene(third, *api.box_scene(500, 1))
hip.host_hip_limit(hip.host_hip_used() + 100 * MB)
try:
    s3.launch(p)
    raise SystemExit("not refused")
except api.VzError as e:
    assert e.status == 2
""")


def test_render_time_holds_no_allocation(stand_in):
    """render_ms runs between two events: the buffers of a launch, of a
    batch's groups and of its large items are there before the first."""
    run(stand_in, """
def check(what):
    log = calls()
    first = log.index("record")
    assert any("k_path" in c for c in log[first:]), what
    late = [c for c in log[first:] if c.startswith(("malloc", "free", "refuse"))]
    assert late == [], (what, late)

calls()
scene.launch(params(64, 36, 2))
check("a first launch")
scene.launch(params(2048, 2048, 131, api.ACCUM_FP64))
check("a launch of several chunks")
t = api.Tuning()
t.queue_capacity = 1 << 20                     # 256 MB: 16M paths
big = [params(1024, 1024, 40), params(2048, 1024, 12, api.ACCUM_FP64), params(4096, 4096, 2)]
api.batch_launch(ctx, [(scene, params(512, 512, 4)), (scene, big[0]), (scene, big[1]), (scene, big[2])], tuning=t)
check("a batch with large items")
""")


def test_kept_memory_is_given_back(stand_in):
    """What a context keeps between calls (blocks of destroyed scenes, launch
    buffers) makes room when one of its allocations fails, whichever it is,
    and goes back when the caller asks."""
    run(stand_in, """
L = api.lib()
base = hip.host_hip_used()

def keep(n=1_000_000):
    api.Scene(ctx, *api.box_scene(n, 1)).close()   # about 350 MB
    assert hip.host_hip_used() > base + 300 * MB

rays = api.RAY_DT
def no_room(f):
    keep()
    hip.host_hip_limit(hip.host_hip_used())
    out = f()
    hip.host_hip_limit(1 << 60)
    assert hip.host_hip_used() < base + 3500 * MB
    return out

buf = C.c_void_p(4096)
st = api.Stats()
no_room(lambda: api.check(L.vzTraceClosest(scene.h, buf, 1000, buf, None, C.byref(st))))
no_room(lambda: scene.launch(params(64, 36, 2, api.MEGAKERNEL)))
no_room(lambda: scene.launch(params(64, 36, 2)))
scene.launch(params(1920, 1080, 64))              # 2.1 GB of launch buffers, kept
hip.host_hip_limit(hip.host_hip_used() + 400 * MB)
big = api.Scene(ctx, *api.box_scene(4_000_000, 1))  # 1.4 GB
big.close()
hip.host_hip_limit(1 << 60)
scene.launch(params(1920, 1080, 64))
t = api.Tuning()
api.batch_launch(ctx, [(scene, params(512, 512, 16))] * 2, tuning=t)
keep()
ctx.trim()
assert hip.host_hip_used() <= base, (hip.host_hip_used(), base)
scene.launch(params(64, 36, 2))                   # and goes on
""")


SERVE = """
class Steps:
    # the flights of a server, finished one at a time
    def __init__(self):
        hip.host_hip_hold(1)

    def settle(self, flights):
        for _ in range(200):
            if hip.host_hip_held() == flights:
                return
            time.sleep(0.01)
        raise AssertionError(f"{hip.host_hip_held()} flights, not {flights}")

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        hip.host_hip_hold(0)
        while hip.host_hip_release():
            pass
"""


def test_small_request_does_not_wait_for_large_ones(stand_in):
    """Two requests of 2.1e9 paths each are running when a thumbnail comes: it
    is rendered within a few launches, long before either is done."""
    run(stand_in, SERVE + """
srv = api.Server(ctx, 8 << 30)
with Steps() as steps:
    large = [srv.submit(scene, params(2048, 2048, 512)) for _ in range(2)]
    steps.settle(2)
    thumb = srv.submit(scene, params(64, 36, 2))
    time.sleep(0.1)
    for turn in range(1, 5):
        assert hip.host_hip_release()
        time.sleep(0.1)
        if srv.poll(thumb) is not None:
            break
    assert srv.poll(thumb) is not None and turn <= 3, turn
    assert [srv.poll(i) for i in large] == [None, None]
srv.drain()
assert all(srv.poll(i).status == 0 for i in large)
assert hip.host_hip_launches(b"k_path_resolve") > 2 * 25    # in slices
srv.close()
""")


def test_server_memory_stays_within_its_budget(stand_in):
    """What a server allocates for its requests is within hbm_budget_bytes
    (beside 2 MB of tables), for budgets from one small request's footprint to
    the default buffers', and each of them is rendered; a request whose own
    footprint is above the budget is refused."""
    run(stand_in, """
TABLES = 2 * MB
small = params(96, 64, 4)
fp = lambda p: api.footprint(p)
assert fp(small) == 96 * 64 * 4 * 16 + 256                      # seeds and radiances of its paths
sliced = params(2048, 2048, 100, api.ACCUM_FP64)                # 6 slices of at most 17 passes
px = 2048 * 2048
assert fp(sliced) == px * 17 * 16 + 256 + px * 28
big = [params(2048, 2048, 7), params(1024, 1024, 64), sliced, params(512, 512, 16), params(1920, 1080, 300)]
mixes = [(fp(small), [small] * 5), (fp(small) * 3 // 2, [small] * 5),
         (max(map(fp, big)), big * 2 + [small] * 20), (3 << 29, big * 3), (2 << 30, big * 4), (64 << 30, big * 2)]
for budget, reqs in mixes:
    for tuning in (None, api.Tuning(queue_capacity=1)):
        base = hip.host_hip_used()
        hip.host_hip_reset_peak()
        srv = api.Server(ctx, budget, tuning=tuning)
        over = srv.submit(scene, params(8192, 8192, 256)) if budget < 4 << 30 else None
        ids = [srv.submit(scene, p) for p in reqs]
        srv.drain()
        assert [srv.poll(i).status for i in ids] == [0] * len(ids), budget
        assert over is None or srv.poll(over).status == 5
        assert hip.host_hip_peak() - base <= budget + TABLES, (budget, tuning, hip.host_hip_peak() - base)
        srv.close()
        assert hip.host_hip_used() <= base
""")


def test_server_short_of_memory_takes_smaller_launches(stand_in):
    """A request alone on a server takes up to 150M paths a launch (2.3 GB),
    for which the two slots of 1.2 GB go.  Where that is not there it goes on
    with the usual 72M, and with less where those are not; the next requests are
    rendered too, also after one that not a single pass of fitted."""
    run(stand_in, """
p = params(2048, 2048, 100)                       # 67 MB a pass, 67 MB carried
for room, launches in ((0, 3), (-600 * MB, 6), (-1400 * MB, 12), (-2150 * MB, 100), (-2200 * MB, 0)):
    srv = api.Server(ctx, 8 << 30)
    hip.host_hip_limit(hip.host_hip_used() + room)
    before = hip.host_hip_launches(b"k_path_resolve")
    i = srv.submit(scene, p)
    srv.drain()
    assert srv.poll(i).status == (0 if launches else 2), room
    done = hip.host_hip_launches(b"k_path_resolve") - before
    j = [srv.submit(scene, params(64, 36, 2)) for _ in range(5)]
    srv.drain()
    assert [srv.poll(k).status for k in j] == [0] * 5
    hip.host_hip_limit(1 << 60)
    srv.close()
    assert done == launches, (room, done)
""")
