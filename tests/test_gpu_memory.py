"""Memory of a renderer's path state (marked gpu): what a sequence of frames
makes it hold, and frames and tuning where the state does not fit.
"""
import ctypes as C
import time

import numpy as np
import pytest

from kuafu_amd import KuafuError, abi, scenes
from kuafu_amd.api import GpuScene, Renderer

pytestmark = pytest.mark.gpu

GIB = 1 << 30


def free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert abi.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def with_lights(w, n):
    """The workload under n lights of all kinds, none of them soft."""
    w.data.point_lights, w.data._n_point = abi.PointLights(), 0
    for k in range(min(n - 1, 32)):
        w.data.add_point_light((4.0 * np.cos(k), 2.0 + 0.05 * k, 4.0 * np.sin(k)), (1, 0.9, 0.8), 3.0, radius=0.0)
    for k in range(n - 33):
        view = scenes.look_at((3.0 * np.cos(2 * k), 4.0, 3.0 * np.sin(2 * k)), (0.0, 0.3, 0.0), (0, 1, 0))
        w.data.add_active_light(view, (0.8, 0.9, 1.0), fov=0.9, strength=20.0)
    return w


def test_paths_and_slots_have_capacities_of_their_own(gpu):
    """4.2 M paths with two lights, then 0.26 M with 41, hold 132 bytes per
    path of the first frame and 69 per path and light of the second: 1.3 GB
    (the product of both, 41 lights for 4.2 M paths, is 12.4)."""
    many, few = scenes.config1(512, 512, spp=16, path_depth=3), with_lights(scenes.config1(512, 512, spp=1, path_depth=3), 41)
    a, b = GpuScene(many.data), GpuScene(few.data)
    r, alone = Renderer(512, 512), Renderer(512, 512)
    alone.render(b, few.cam, few.pc, seed=1)
    want = alone.read(0)
    alone.close()
    before = free_bytes()
    r.render(a, many.cam, many.pc, seed=1, samples_per_batch=16)
    r.render(b, few.cam, few.pc, seed=1)
    assert before - free_bytes() < 2 * GIB
    assert np.array_equal(r.read(0), want)


# 4.2 M pixels at 16 samples: 67 M paths of 270 bytes, and, with 684 bytes
# each, as many as stay within 32 GiB.
@pytest.mark.parametrize("lights,batches", [(2, 1), (8, 2)])
def test_default_batch_by_the_state_of_its_paths(gpu, lights, batches):
    w = with_lights(scenes.config1(2048, 2048, spp=16, path_depth=1), lights)
    gs, r = GpuScene(w.data), Renderer(2048, 2048)
    r.render(gs, w.cam, w.pc, samples_per_batch=1)  # targets, camera rays' tree
    before = free_bytes()
    st = r.render(gs, w.cam, w.pc)
    assert before - free_bytes() < 32 * GIB
    assert st.shadow_launches == 2 * batches
    r.close()


@pytest.fixture
def scarce(gpu):
    """scarce(n): leaves n bytes of GPU memory free until the test ends."""
    L, held = abi.lib(), []
    small = scenes.config1(32, 32, spp=1, path_depth=6)
    gs, r = GpuScene(small.data), Renderer(32, 32)
    for tail in (1, 2, 7):  # code and scratch of the kernels, while there is room
        r.set_schedule(tail_bounce=tail)
        r.render(gs, small.cam, small.pc)

    def leave(n):
        p = C.c_void_p()
        assert L.hipMalloc(C.byref(p), C.c_size_t(free_bytes() - n)) == 0
        held.append(p)

    yield leave
    for p in held:
        assert L.hipFree(p) == 0


def test_default_batch_in_scarce_memory(scarce):
    """A default batch leaves a quarter of the free memory to others, also on
    the frames after the first, which allocate nothing.  33.5 M paths with two
    lights are 9.1 GB: less than three quarters of what is free, more than
    that, and more than is free."""
    w = scenes.config1(2048, 1024, spp=16, path_depth=2)
    gs, ref = GpuScene(w.data), Renderer(2048, 1024)
    ref.render(gs, w.cam, w.pc, seed=1, samples_per_batch=1)
    want = ref.read(0)
    ref.close()
    for free, halved in ((16, False), (10, True), (6, True)):
        scarce(free * GIB)
        r = Renderer(2048, 1024)
        before = free_bytes()
        launches, ms = [], []
        for _ in range(4):
            t = time.perf_counter()
            launches.append(r.render(gs, w.cam, w.pc, seed=1).extend_launches)
            ms.append(time.perf_counter() - t)
            assert free_bytes() >= before // 4 - GIB // 2  # targets, camera rays' tree
        assert len(set(launches)) == 1
        assert np.array_equal(r.read(0), want)
        t = time.perf_counter()
        st = r.render(gs, w.cam, w.pc, seed=1, samples_per_batch=8)
        t = time.perf_counter() - t
        assert (launches[0] > st.extend_launches // 2) == halved
        assert min(ms[1:]) < 5 * t  # 313 ms against 16 where every frame allocated
        r.close()


def test_autotune_in_scarce_memory(scarce):
    """Tuning passes over batches that do not fit (16 samples: 9.1 GB of 6
    GiB), and the renderer draws with what it picked."""
    w = scenes.config1(2048, 1024, spp=16, path_depth=2)
    gs = GpuScene(w.data)
    scarce(6 * GIB)
    r = Renderer(2048, 1024)
    want = r.render(gs, w.cam, w.pc, seed=1, samples_per_batch=1) and r.read(0)
    t = r.autotune(gs, w.cam, w.pc)
    assert 1 <= t["samples_per_batch"] < 16 and t["frame_ms"] < np.inf
    r.render(gs, w.cam, w.pc, seed=1)
    assert np.array_equal(r.read(0), want)


def test_failed_autotune_keeps_the_schedule(gpu):
    w = scenes.config1(64, 64, spp=8, path_depth=4)
    gs, r = GpuScene(w.data), Renderer(64, 64)
    r.set_schedule(samples_per_batch=2, tail_bounce=3)
    before = r.render(gs, w.cam, w.pc).extend_launches
    deep = scenes.config1(64, 64, spp=8, path_depth=70)
    with pytest.raises(KuafuError, match="depth"):
        r.autotune(gs, deep.cam, deep.pc)
    assert r.render(gs, w.cam, w.pc).extend_launches == before == 4 * 3


def test_a_scene_does_not_keep_its_largest_ray_batch(gpu):
    """A batch of 1 M rays (59 MB of rays and hits) leaves a scene with the 16
    MiB at most that smaller batches keep."""
    gs = GpuScene(scenes.config1().data)
    rng = np.random.default_rng(3)
    rays = np.zeros(1 << 20, abi.RAY_DTYPE)
    rays["org"], rays["tmax"] = rng.uniform(-2, 2, (len(rays), 3)), 10.0
    rays["dir"] = rng.normal(size=(len(rays), 3))
    few = gs.trace_closest(rays[:1000])  # pinned memory, counters
    before = free_bytes()
    for n in (1 << 20, 1 << 18, 400000):
        assert gs.trace_closest(rays[:n])[:1000].tobytes() == few.tobytes()
        assert before - free_bytes() <= 16 << 20
