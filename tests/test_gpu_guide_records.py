"""The training kernel at the edges of its record tiles (32 records a wave, 256 a
block, a second group per block above 65536) and of the record upload.

  - records of weight zero add nothing: a gradient over n records and one over
    2n, the second half of weight zero and the first of twice the weight, are
    equal bit for bit (the factors are powers of two, the sums keep their order);
  - against the oracle: loss within 1e-3, every layer's gradient within 1e-2 in
    relative L2 norm (BF16 operands, the bar of the gradient test)."""
import numpy as np
import pytest

import wurstrenderer_amd as wr
from oracle import guide as G
from test_gpu_guide import guide_scene, params, records, scene_box  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 255, 256, 257, 8191])
def test_records_of_weight_zero_add_nothing(guide_scene, n):  # noqa: F811
    sc, gs = guide_scene
    print(f"guide gradient: {n} records and {2 * n} with half of them weightless", flush=True)
    g = wr.Guide(gs)
    rng = np.random.default_rng(n)
    g.set_params(params(rng, scale_out=1.0))
    pos, nrm, wo, wi, w = records(rng, 2 * n, scene_box(sc))
    _, a = g.gradient(pos[:n], nrm[:n], wo[:n], wi[:n], w[:n])
    w2 = np.concatenate([2 * w[:n], np.zeros_like(w[n:])])
    _, b = g.gradient(pos, nrm, wo, wi, w2)
    assert np.any(a != 0) and np.array_equal(a, b)


@pytest.mark.parametrize("n", [257, 65536 + 33])
def test_gradient_over_several_groups_matches_oracle(guide_scene, n):  # noqa: F811
    sc, gs = guide_scene
    print(f"guide gradient: {n} records against the oracle", flush=True)
    g = wr.Guide(gs)
    rng = np.random.default_rng(n)
    p = params(rng, scale_out=1.0)
    g.set_params(p)
    rec = records(rng, n, scene_box(sc))
    loss, grad = g.gradient(*rec)
    rloss, rgrad = G.loss_and_grad(p, *rec, scene_box(sc), bf=True)
    assert abs(loss - rloss) < 1e-3 * abs(rloss)
    o = 0
    for k, m in G.SHAPES:
        for sz in (k * m, m):
            a, b = grad[o:o + sz], rgrad[o:o + sz]
            assert np.linalg.norm(a - b) < 1e-2 * np.linalg.norm(b)
            o += sz
