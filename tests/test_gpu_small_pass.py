"""Passes of few samples, which one kernel renders from start to end, against the
same passes through the path queues (a path pool one smaller than the pass).

Both do the same arithmetic on each sample and sum it in the same order, so base
films are equal bit for bit and ray counts are equal; the splat film is FP64
atomics in varying order and agrees to rounding (1e-11).  Sizes: one pixel, edges
of the 64-path tiles, several samples per pixel, shares that restart lanes (above
2^18 samples), and both sides of the limits (2^22 samples up to 2^11 triangles,
2^20 up to 2^16, else 2^18)."""
import ctypes as C

import numpy as np
import pytest

import wurstrenderer_amd as wr
from wurstrenderer_amd import scenes

pytestmark = pytest.mark.gpu

SCENES = {
    "cornell": lambda r: scenes.cornell(1, resolution=r),
    "spheres": lambda r: scenes.icospheres(2, n_spheres=12, level=3, resolution=r),
    "env": lambda r: scenes.icospheres(2, n_spheres=12, level=3, resolution=r).with_envmap((0.3, 0.4, 0.5)),
    "clutter": lambda r: scenes.cornell_clutter(3, 12_000, r),
    "room": lambda r: scenes.guide_room(4, n_spheres=49, level=4, resolution=r),
}


def _films(gs, render, total, spp, **kw):
    out = []
    for pool in (0, total - 1):
        f = wr.Film(gs)
        st = render(gs, f, spp, seed=9, max_paths_in_flight=pool, **kw)
        out.append((*f.read(), st.extend_rays, st.shadow_rays, st.paths))
        f.close()
    return out


@pytest.mark.parametrize("kind", list(SCENES))
@pytest.mark.parametrize("size,spp,vertices", [((1, 2), 1, 8), ((9, 7), 1, 2), ((64, 1), 1, 3), ((13, 5), 1, 8), ((63, 65), 3, 10),
                                               ((512, 512), 1, 12), ((512, 513), 1, 6),
                                               ((1024, 1024), 1, 9), ((1024, 1025), 1, 4)])
def test_small_passes_equal_the_queues(gpu_device, kind, size, spp, vertices):
    print(f"small pass: {kind} {size} spp={spp} N={vertices}", flush=True)
    gs = wr.GpuScene(gpu_device, SCENES[kind](size))
    total = size[0] * size[1] * spp
    for render, kw in ((wr.render_nee, {}), (wr.render_nee, dict(use_mis=False)), (wr.render_primitive, {})):
        a, b = _films(gs, render, total, spp, num_path_vertices=vertices, **kw)
        np.testing.assert_array_equal(a[0], b[0])
        np.testing.assert_allclose(a[1], b[1], rtol=1e-11, atol=1e-300)
        assert a[2:] == b[2:]


@pytest.mark.parametrize("vertices", [255, 256, 300])
def test_more_vertices_than_the_bounce_counter_holds(gpu_device, vertices):
    """Above 255 vertices the queues render the pass, which bound the iterations
    of paths that the 8-bit bounce counter would never end (open scene: all end)."""
    print(f"small pass: spheres, {vertices} vertices", flush=True)
    gs = wr.GpuScene(gpu_device, SCENES["spheres"]((33, 17)))
    a, b = _films(gs, wr.render_nee, 33 * 17, 1, num_path_vertices=vertices)
    np.testing.assert_array_equal(a[0], b[0])
    assert a[2:] == b[2:]


@pytest.mark.parametrize("spp", [16, 17])
def test_shares_up_to_the_limit_of_a_tiny_scene(gpu_device, spp):
    print(f"small pass: cornell 512x512 spp={spp}", flush=True)
    gs = wr.GpuScene(gpu_device, SCENES["cornell"]((512, 512)))
    a, b = _films(gs, wr.render_nee, 512 * 512 * spp, spp, num_path_vertices=12)
    np.testing.assert_array_equal(a[0], b[0])
    assert a[2:] == b[2:]


def test_small_pass_in_the_fixed_region(gpu_device):
    """The allocation-free entry point: 32,768 samples fit its spill slices, 33,024 take the queues."""
    for size in ((256, 128), (256, 129)):
        print(f"small pass, fixed region: {size}", flush=True)
        gs = wr.GpuScene(gpu_device, SCENES["spheres"](size))
        a, b = wr.Film(gs), wr.Film(gs)
        wr.render_nee(gs, a, 1, num_path_vertices=8, seed=3)
        prm, st = wr.render_params(1, 8, 3), wr.RenderStats()
        assert wr.lib().wr_render_nee_noalloc(gs.h, b.h, C.byref(prm), C.byref(st)) == 0
        np.testing.assert_array_equal(a.read()[0], b.read()[0])
