"""Passes with fewer samples than the path pool holds.

From their first iteration on, most blocks of the shade kernels have no work, and
the last of them to finish ends the iteration.  The same render through a pool
smaller than its last pass keeps every block busy; base films are equal bit for
bit (a sample's radiance does not depend on the pool, and samples are summed in
order), ray counts are equal, and the splat film, FP64 atomics in varying order,
agrees to rounding: at most 10^4 terms of 1.1e-16 per pixel."""
import ctypes as C

import numpy as np
import pytest

import wurstrenderer_amd as wr
from wurstrenderer_amd import scenes

pytestmark = pytest.mark.gpu


# samples of a pass: 2^27 (1,024 of 1,025 per pixel), 3 per pixel (of 4), 2^20 (11 of 12 per pixel)
@pytest.mark.parametrize("kind,size,pools", [("nee", (512, 256), (1 << 18, 100_000)), ("light", (512, 256), (1 << 18, 100_000)),
                                             ("guided", (512, 256), (0, 100_000)), ("fixed", (300, 300), (1 << 17, 60_000))])
def test_last_pass_smaller_than_the_pool(gpu_device, kind, size, pools):
    gs = wr.GpuScene(gpu_device, scenes.icospheres(2, n_spheres=12, level=3, resolution=size))
    guide = wr.Guide(gs) if kind == "guided" else None
    want = None
    for pool in pools:
        print(f"last pass: {kind} pool={pool}", flush=True)
        film = wr.Film(gs)
        common = dict(num_path_vertices=4, seed=6, max_paths_in_flight=pool)
        if kind == "nee":  # counting keeps the last pass in the queues
            st = wr.render_nee(gs, film, 1025, count_traversal=True, **common)
        elif kind == "light":
            st = wr.render_light(gs, film, 1025, **common)
        elif kind == "guided":
            st, _ = wr.render_guided(gs, film, guide, 4, guide_fraction=0.3, spp_per_pass=3, train_steps=0,
                                     warmup_passes=0, **common)
        else:
            prm, st = wr.render_params(12, **common), wr.RenderStats()
            assert wr.lib().wr_render_nee_noalloc(gs.h, film.h, C.byref(prm), C.byref(st)) == 0
        got = (*film.read(), st.extend_rays, st.shadow_rays)
        film.close()
        if want is None:
            want = got
            assert got[1 if kind == "light" else 0].any()
        np.testing.assert_array_equal(got[0], want[0])
        np.testing.assert_allclose(got[1], want[1], rtol=1e-11, atol=1e-300)
        assert got[2:] == want[2:]
