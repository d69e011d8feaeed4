"""The shade kernels' block sizes and their combined append.

The pool size sets the threads per block (64 to 512 by powers of two on a
256-CU device) and with it which path lands where in the queues.  A sample's
radiance does not depend on either and the base film sums samples in order, so
base films are equal bit for bit across pools; the splat film is FP64 atomics
in varying order and agrees to rounding.  The ray counts are equal."""
import numpy as np
import pytest

import wurstrenderer_amd as wr
from wurstrenderer_amd import scenes

pytestmark = pytest.mark.gpu

# 256 x 256 at 8 spp = 524,288 samples, one pass: blocks of 64 (with 512 refills), 64, 128, 256, 512, 512 threads
POOLS = [1024, 65_535, 65_536, 140_001, 262_144, 0]


def _scene(kind):
    if kind == "fog":
        return scenes.cornell_clutter(3, 12_000, (256, 256)).with_medium(sigma_a=0.05, sigma_s=0.4, g=0.7)
    sc = scenes.icospheres(2, n_spheres=12, level=3, resolution=(256, 256))
    return sc.with_envmap((0.3, 0.4, 0.5)) if kind == "env" else sc


@pytest.mark.parametrize("kind", ["nee", "env", "fog", "light"])
def test_films_do_not_depend_on_the_pool(gpu_device, kind):
    gs = wr.GpuScene(gpu_device, _scene(kind))
    render = wr.render_light if kind == "light" else wr.render_nee
    want = None
    for pool in POOLS:
        film = wr.Film(gs)
        st = render(gs, film, 8, num_path_vertices=8, seed=4, max_paths_in_flight=pool)
        base, splat = film.read()
        print(f"shade blocks: {kind} pool={pool} rays={st.extend_rays}+{st.shadow_rays}", flush=True)
        if want is None:
            want = (base, splat, st.extend_rays, st.shadow_rays)
            assert splat.any() if kind == "light" else base.any()
        np.testing.assert_array_equal(base, want[0])
        np.testing.assert_allclose(splat, want[1], rtol=1e-11, atol=1e-300)
        assert (st.extend_rays, st.shadow_rays) == want[2:]
