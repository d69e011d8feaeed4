"""Host transfers through the pinned ring: film reads, device-composed images
and ray batches at the sizes where the chunking can go wrong (one value, one
below and above a 1 MB chunk, several threads with a ragged last chunk).

The copies are exact and the image is the same FP64 divisions and addition on
the device as in numpy, so everything is compared bit for bit."""
import threading

import numpy as np
import pytest

import wurstrenderer_amd as wr
from wurstrenderer_amd import scenes

pytestmark = pytest.mark.gpu
CHUNK_VALUES = (1 << 20) // 8


# 3 W H values: 3; just below and above one chunk; 3 MB and 7.5 chunks (threads); 26 chunks
@pytest.mark.parametrize("size", [(1, 1), (209, 209), (211, 209), (410, 320), (641, 511), (1100, 1031)])
def test_film_image_equals_numpy(gpu_device, size):
    gs = wr.GpuScene(gpu_device, scenes.cornell(1, resolution=size))
    film = wr.Film(gs)
    wr.render_nee(gs, film, 3, num_path_vertices=4, seed=2)
    base, splat = film.read()
    print(f"image: {size} values={base.size} chunks={base.size / CHUNK_VALUES:.2f}", flush=True)
    assert base.shape == (size[1], size[0], 3) and (size == (1, 1) or (base.any() and splat.any()))
    W, H = size
    np.testing.assert_array_equal(film.image(), base / film.spp + splat / (film.spp * W * H))


@pytest.mark.parametrize("n", [1, 63, 65, 32768, 32769, 262144, 262145, 800_001])
def test_ray_batches_do_not_depend_on_their_size(gpu_device, n):
    sc = scenes.icospheres(2, n_spheres=6, level=3, resolution=(8, 8))
    gs = wr.GpuScene(gpu_device, sc)
    rays = np.concatenate([scenes.random_rays(sc, (n + 1) // 2, seed=1), scenes.random_rays(sc, n // 2, seed=2, inside=True)])
    rng = np.random.default_rng(5)
    rays = np.ascontiguousarray(rays[rng.permutation(n)])
    rays[:, 7] = np.where(rng.random(n) < 0.5, np.inf, rng.uniform(0.5, 20.0, n))
    g, p, t = gs.trace_closest(rays)
    occ = gs.trace_any(rays)
    print(f"rays: {n}", flush=True)
    np.testing.assert_array_equal(occ.astype(bool), g != 0xFFFFFFFF)
    np.testing.assert_array_equal(np.isinf(t), g == 0xFFFFFFFF)
    pick = np.unique(np.concatenate([np.arange(min(n, 50)), np.arange(max(0, n - 50), n), rng.integers(0, n, 400)]))
    g1, p1, t1 = gs.trace_closest(np.ascontiguousarray(rays[pick]))
    np.testing.assert_array_equal(g[pick], g1)
    np.testing.assert_array_equal(p[pick], p1)
    np.testing.assert_array_equal(t[pick], t1)


def test_transfers_from_several_threads(gpu_device):
    """Two scenes of one device, each read by its own thread at the same time."""
    work = []
    for k in range(2):
        gs = wr.GpuScene(gpu_device, scenes.cornell(k + 1, resolution=(700, 500 + k)))
        film = wr.Film(gs)
        wr.render_nee(gs, film, 2, num_path_vertices=3, seed=k)
        work.append((gs, film, film.image()))
    bad = []

    def read(film, want):
        for _ in range(5):
            if not np.array_equal(film.image(), want):
                bad.append(film)

    threads = [threading.Thread(target=read, args=(f, im)) for _, f, im in work]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad
