"""Records of up to what the pinned ring holds (322,638) go up without a wait of their
own, in chunks of 20,164, more of them through the ring's slots in turn.  Weightless records add nothing and the factors are
powers of two, so a gradient over n records equals one over 2n bit for bit."""
import threading

import numpy as np
import pytest

import wurstrenderer_amd as wr
from test_gpu_guide import guide_scene, params, records, scene_box  # noqa: F401
from wurstrenderer_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 10_083, 20_164, 20_165])
def test_both_routes_of_an_upload(guide_scene, n):  # noqa: F811
    sc, gs = guide_scene
    print(f"record upload: {n} and {2 * n}", flush=True)
    g = wr.Guide(gs)
    rng = np.random.default_rng(n)
    g.set_params(params(rng, scale_out=1.0))
    pos, nrm, wo, wi, w = records(rng, 2 * n, scene_box(sc))
    _, a = g.gradient(pos[:n], nrm[:n], wo[:n], wi[:n], w[:n])
    _, b = g.gradient(pos, nrm, wo, wi, np.concatenate([2 * w[:n], np.zeros_like(w[n:])]))
    assert np.any(a != 0) and np.array_equal(a, b)


def test_training_and_transfers_of_several_threads(gpu_device):
    """Two threads train and one reads images, all through the ring of one device."""
    sc = scenes.cornell(1, resolution=(300, 200))
    scs = [wr.GpuScene(gpu_device, sc) for _ in range(3)]
    film = wr.Film(scs[2])
    wr.render_nee(scs[2], film, 1, num_path_vertices=4, seed=1)
    want_image = film.image()
    rng = np.random.default_rng(5)
    p0 = params(rng, scale_out=1.0)
    rec = records(rng, 3000, scene_box(sc))
    guides = [wr.Guide(s) for s in scs[:2]]
    guides[0].set_params(p0)
    guides[0].train(*rec, steps=5)
    want, bad = guides[0].get_params(), []

    def train(g):
        for _ in range(10):
            g.set_params(p0)
            g.train(*rec, steps=5)
            if not np.array_equal(g.get_params(), want):
                bad.append("params")

    def read():
        for _ in range(30):
            if not np.array_equal(film.image(), want_image):
                bad.append("image")

    threads = [threading.Thread(target=train, args=(g,)) for g in guides] + [threading.Thread(target=read)]
    [t.start() for t in threads]
    [t.join(60) for t in threads]
    assert not bad and not any(t.is_alive() for t in threads)


@pytest.mark.parametrize("n", [322_638, 322_639, 400_000])
def test_uploads_around_the_size_of_the_ring(guide_scene, n):  # noqa: F811
    """The last 4,096 records count and the rest are weightless, so the sums are those
    of a gradient over the 4,096 alone, FP32 sums of the same products in another order
    (the bars of the gradient test: loss 1e-3, gradient 1e-2 in relative L2 norm)."""
    sc, gs = guide_scene
    print(f"record upload: {n}", flush=True)
    g = wr.Guide(gs)
    rng = np.random.default_rng(n)
    g.set_params(params(rng, scale_out=1.0))
    few = records(rng, 4096, scene_box(sc))
    pos, nrm, wo, wi = (np.resize(a, (n, 3)) for a in few[:4])
    w = np.zeros(n, np.float32)
    w[-4096:] = np.resize(few[4], n)[-4096:]
    last = [np.ascontiguousarray(a[-4096:]) for a in (pos, nrm, wo, wi, w)]
    loss, grad = g.gradient(pos, nrm, wo, wi, w)
    loss1, grad1 = g.gradient(*last)
    # means over n and over 4,096 records
    np.testing.assert_allclose(loss * n, loss1 * 4096, rtol=1e-4)
    a, b = grad * np.float32(n), grad1 * np.float32(4096)
    assert np.linalg.norm(a - b) < 1e-2 * np.linalg.norm(b)
