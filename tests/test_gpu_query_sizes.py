"""Ray queries and film reads at the sizes where their route changes.

Rays: up to 32,768 are read from pinned memory by the kernel; up to 1,310,720 hits
and 15,728,640 flags are written there.  Films: arrays up to 16 KB and from 1.2 MB
on (26^2 and 27^2, 223^2 and 224^2 pixels) come through the pinned ring, those in
between by plain copies.  Everything is exact, so comparisons are too."""
import threading
import time

import numpy as np
import pytest

import wurstrenderer_amd as wr
from wurstrenderer_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 32_767, 32_768, 32_769, 87_382, 349_526, 1_310_720, 1_310_721])
def test_hits_equal_those_of_parts(gpu_device, n):
    """A query gives what the same rays give in pieces of 10,007."""
    print(f"query: {n} rays", flush=True)
    sc = scenes.icospheres(2, n_spheres=6, level=3, resolution=(8, 8))
    gs = wr.GpuScene(gpu_device, sc)
    rays = np.concatenate([scenes.random_rays(sc, (n + 1) // 2, seed=1), scenes.random_rays(sc, n // 2, seed=2, inside=True)])
    rays[:, 7] = np.where(np.arange(n) % 3 == 0, 4.0, np.inf)
    whole, flags = gs.trace_closest(rays), gs.trace_any(rays)
    for at in range(0, n, 10_007):
        part = rays[at:at + 10_007]
        for a, b in zip(whole, gs.trace_closest(part)):
            np.testing.assert_array_equal(a[at:at + 10_007], b)
        np.testing.assert_array_equal(flags[at:at + 10_007], gs.trace_any(part))
    assert 0 < flags.sum() < n or n == 1


def test_flags_above_the_pinned_limit(gpu_device):
    n = 15 * (1 << 20) + 1
    print(f"query: {n} flags", flush=True)
    sc = scenes.cornell(1, (8, 8))
    gs = wr.GpuScene(gpu_device, sc)
    part = scenes.random_rays(sc, 30_011, seed=3)
    part[:, 7] = 3.0
    rays = np.resize(part, (n, 8))
    want = gs.trace_any(part)
    for m in (n - 1, n):
        np.testing.assert_array_equal(gs.trace_any(rays[:m]), np.resize(want, m))


@pytest.mark.parametrize("size", [1, 26, 27, 40, 223, 224, 361])
def test_film_reads_equal_single_arrays(gpu_device, size):
    print(f"film read: {size}", flush=True)
    gs = wr.GpuScene(gpu_device, scenes.cornell(1, (size, size)))
    film = wr.Film(gs)
    wr.render_nee(gs, film, 2, num_path_vertices=4, seed=1)
    base, splat = film.read()
    alone = np.empty_like(base)
    for want, args in ((base, (alone.ctypes.data, None)), (splat, (None, alone.ctypes.data))):
        alone[:] = -1.0
        assert wr.lib().wr_film_read(film.h, *args) == 0
        np.testing.assert_array_equal(alone, want)
    np.testing.assert_array_equal(film.image(), base / 2 + splat / (2 * size * size))


def _shortest(call, times):
    best = np.inf
    for _ in range(times):
        t = time.perf_counter()
        call()
        best = min(best, time.perf_counter() - t)
    return best


def test_a_small_query_is_one_launch_and_one_wait(gpu_device):
    """1,000 hits take 28 us and a plain copy of 31 KB (Guide.get_params) 13 us; with
    a wait for each array's own transfer the query took 102, with two waits and the
    host's lookup 61.  Shortest of many, so that other load does not count."""
    sc = scenes.cornell(1, (8, 8))
    gs = wr.GpuScene(gpu_device, sc)
    guide = wr.Guide(gs)
    rays = scenes.random_rays(sc, 1000, seed=1)
    query, copy = _shortest(lambda: gs.trace_closest(rays), 300), _shortest(guide.get_params, 300)
    print(f"query {query * 1e6:.1f} us, copy {copy * 1e6:.1f} us", flush=True)
    assert query < 4 * copy


def test_uploads_grow_evenly_with_their_size(gpu_device):
    """Gradients of 60,000 and 80,000 records (3.1 and 4.2 MB up): the larger takes at
    most 4/3 of the smaller (and 5%), where threads started for it made it 1.5 at best
    and 2.3 at the median (278 us and 650)."""
    sc = scenes.cornell(1, (8, 8))
    guide = wr.Guide(wr.GpuScene(gpu_device, sc))
    rng = np.random.default_rng(1)

    def records(n):
        v = rng.normal(size=(4, n, 3)).astype(np.float32)
        v[1:] /= np.linalg.norm(v[1:], axis=2, keepdims=True)
        return (*v, np.ones(n, np.float32))

    times = []
    for n in (60_000, 80_000):
        r = records(n)
        times.append(_shortest(lambda: guide.gradient(*r), 100))
        print(f"gradient of {n}: {times[-1] * 1e6:.0f} us", flush=True)
    assert times[1] < 1.4 * times[0]


def test_queries_of_several_threads(gpu_device):
    """Four scenes of one device, queried at the same time: some calls find the pinned
    ring free and some do not, and all answer what they answer alone."""
    print("queries of several threads", flush=True)
    work, bad = [], []
    for k, n in enumerate((1000, 30_000, 40_000, 1_400_000)):
        sc = scenes.icospheres(2 + k, n_spheres=6, level=3, resolution=(8, 8))
        gs = wr.GpuScene(gpu_device, sc)
        rays = scenes.random_rays(sc, n, seed=k)
        work.append((gs, rays, gs.trace_closest(rays), gs.trace_any(rays)))

    def query(gs, rays, hits, flags):
        for _ in range(400_000 // len(rays) + 2):
            if not all(np.array_equal(a, b) for a, b in zip(gs.trace_closest(rays), hits)):
                bad.append(len(rays))
            if not np.array_equal(gs.trace_any(rays), flags):
                bad.append(len(rays))

    threads = [threading.Thread(target=query, args=w) for w in work]
    [t.start() for t in threads]
    [t.join(60) for t in threads]
    assert not bad and not any(t.is_alive() for t in threads)
