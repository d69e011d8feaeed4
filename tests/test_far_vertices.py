"""Scenes with a vertex so far out that box areas overflow FP32 (from about 1e19 on).
Every finite vertex is accepted, so the builders must still make a valid tree: a
subtree of more triangles than a leaf holds stays a subtree, whatever its cost."""
import dataclasses

import numpy as np
import pytest

import wurstrenderer_amd as wr
from wurstrenderer_amd import scenes

FAR = [1e15, 3e18, 2e19, 1e20, 1e25, 1e30, 3e33, 1e34, 1e36, 1e38]


def far_scene(far, sides=(1, 1, 1), near=None):
    """A small scene and, behind its geometries, a triangle that reaches out to `far` on each axis."""
    sc = near if near is not None else scenes.icospheres(2, n_spheres=4, level=2, resolution=(8, 8))
    a = np.float32(far) * np.asarray(sides, np.float32)
    verts = np.concatenate([sc.verts, [a, a * np.float32([1, 0.5, 1]), a * np.float32([1, 1, 0.5])]]).astype(np.float32)
    nv = len(sc.verts)
    return dataclasses.replace(sc, verts=verts, tris=np.concatenate([sc.tris, [[nv, nv + 1, nv + 2]]]).astype(np.uint32),
                               tri_geom=np.append(sc.tri_geom, len(sc.geom_material)).astype(np.uint32),
                               geom_material=np.append(sc.geom_material, 0).astype(np.int32),
                               geom_light=np.append(sc.geom_light, -1).astype(np.int32))


@pytest.mark.parametrize("far", FAR)
def test_host_tree_is_valid(far):
    wr.bvh_selftest(far_scene(far))
    wr.bvh_selftest(far_scene(-far))


@pytest.mark.gpu
@pytest.mark.parametrize("far", FAR)
@pytest.mark.parametrize("builder", ["gpu", "host"])
def test_device_tree_is_valid(gpu_device, builder, far):
    print(f"far vertices: {builder} {far}", flush=True)
    for sc in (far_scene(far), far_scene(-far)):
        gs = wr.GpuScene(gpu_device, sc, builder=builder)
        gs.bvh_check(sc)


@pytest.mark.gpu
@pytest.mark.parametrize("far", FAR)
@pytest.mark.parametrize("builder", ["gpu", "host"])
def test_near_triangles_are_hit_whatever_lies_far_out(gpu_device, builder, far):
    """Rays between the near triangles find in the large scene what they find without
    the far triangle, in every octant of directions: where the planes of all three axes
    overflow, a box is entered and not passed over.  (The same triangle test on the same
    vertices, so distances are equal; a ray that finds nothing near may hit the far one.)"""
    near = scenes.triangle_soup(800, seed=5)
    rays = scenes.random_rays(near, 16_000, seed=3, inside=True)
    octants = np.array([[1 - 2 * (k >> b & 1) for b in range(3)] for k in range(8)], np.float32)
    rays[:, 4:7] = np.abs(rays[:, 4:7]) * octants[np.arange(len(rays)) % 8]
    alone = wr.GpuScene(gpu_device, near, builder=builder)
    g0, _, t0 = alone.trace_closest(rays)
    hit = g0 != 0xFFFFFFFF
    assert all(hit[k::8].sum() > 50 for k in range(8))
    for sides in ((1, 1, 1), (-1, -1, -1), (1, -1, 1)):
        sc = far_scene(far, sides, near)
        gs = wr.GpuScene(gpu_device, sc, builder=builder)
        gs.bvh_check(sc)  # every ref is a node or a leaf: the traversal ends
        print(f"far vertices: {builder} {far} {sides}", flush=True)
        g, _, t = gs.trace_closest(rays)
        np.testing.assert_array_equal(t[hit], t0[hit])
        np.testing.assert_array_equal(g[hit], g0[hit])
        short = rays.copy()
        short[:, 7] = np.where(hit, t0 * np.float32(1.01), 1.0)
        assert gs.trace_any(short)[hit].all()


@pytest.mark.gpu
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_rays_that_are_not_finite_miss_at_the_root(gpu_device, value):
    """One component or all of an origin or a direction; the finite rays between them
    keep their hits, and a wave of such rays costs what a wave of misses costs, not
    the whole tree (300,000 nodes one after the other, a microsecond each)."""
    import time

    print(f"rays that are not finite: {value}", flush=True)
    sc = scenes.icospheres(2, n_spheres=64, level=5, resolution=(8, 8))
    gs = wr.GpuScene(gpu_device, sc)
    rays = scenes.random_rays(sc, 640, seed=3)
    want = gs.trace_closest(rays)
    assert (want[0] != 0xFFFFFFFF).sum() > 50
    broken = np.arange(640) % 5 == 0
    for where in ([0], [0, 1, 2], [4], [6], [4, 5, 6], [0, 1, 2, 4, 5, 6]):
        r = rays.copy()
        r[np.ix_(broken, where)] = value
        g, p, t = gs.trace_closest(r)
        assert (g[broken] == 0xFFFFFFFF).all() and np.isinf(t[broken]).all() and not gs.trace_any(r)[broken].any()
        for a, b in zip((g, p, t), want):
            np.testing.assert_array_equal(a[~broken], b[~broken])
        start = time.perf_counter()
        gs.trace_closest(r)
        assert time.perf_counter() - start < 0.02
