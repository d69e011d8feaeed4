"""The GPU scene build where its parts meet: cluster counts around the capacity
of the one-block clustering kernel, mesh checks on the device, and builds that
share the device handle's memory.

  - every tree passes the builder's invariant checks, two builds of a scene are
    byte-identical, and the closest hits of a ray set are those of the
    host-built tree: t within 1e-5 t (the FP32 watertight test), bit-identical
    for at least 99.9% of the rays;
  - a faulty mesh is refused with the error code and message of the host-side
    check, wherever in the arrays the fault is, and the next build succeeds;
  - builds from four threads on one device handle give the serial hash."""
import dataclasses
import threading

import numpy as np
import pytest

import wurstrenderer_amd as wr
from wurstrenderer_amd import scenes

pytestmark = pytest.mark.gpu


def _soup(n, copies=1, seed=3):
    rng = np.random.default_rng(seed)
    v = rng.uniform(-1, 1, (n // copies, 1, 3)) + 0.1 * rng.normal(size=(n // copies, 3, 3))
    v = np.concatenate([np.repeat(v, copies, axis=0), v[:n % copies]]).reshape(-1, 3)
    b = scenes.SceneBuilder()
    m = b.material(scenes.LAMBERT, rho_d=(0.5, 0.5, 0.5))
    half = n // 2
    if half:
        b.mesh(v[:3 * half], np.arange(3 * half).reshape(-1, 3), material=m)
    b.mesh(v[3 * half:], np.arange(3 * (n - half)).reshape(-1, 3), material=m)
    return b.build(dict(pos=(0, 0, 8), lookat=(0, 0, 0), fovy=45.0, resolution=(8, 8)), name=f"soup{n}x{copies}")


@pytest.mark.parametrize("n,copies", [(1, 1), (2, 1), (3, 1), (65, 1), (2047, 1), (2048, 1), (2049, 1), (2500, 5),
                                      (4097, 1), (9001, 3)])
def test_clustering_around_the_one_block_limit(gpu_device, n, copies):
    sc = _soup(n, copies)
    print(f"build: {sc.name}", flush=True)
    a, b = wr.GpuScene(gpu_device, sc), wr.GpuScene(gpu_device, sc)
    sa, sb = a.bvh_check(sc), b.bvh_check(sc)
    assert sa["hash"] == sb["hash"]
    h = wr.GpuScene(gpu_device, sc, builder="host")
    rays = scenes.random_rays(sc, 4000, seed=5)
    tg, th = a.trace_closest(rays)[2], h.trace_closest(rays)[2]
    hit = np.isfinite(th) & (th < 1e30)
    np.testing.assert_allclose(tg[hit], th[hit], rtol=1e-5)
    assert np.mean(tg == th) >= 0.999


def _bad(sc, what):
    sc = dataclasses.replace(sc, verts=sc.verts.copy(), tris=sc.tris.copy(), tri_geom=sc.tri_geom.copy())
    if what == "nan_first":
        sc.verts[0, 0] = np.nan
    elif what == "inf_last":
        sc.verts[-1, 2] = -np.inf
    elif what == "index_last":
        sc.tris[-1, 2] = len(sc.verts)
    elif what == "index_max":
        sc.tris[0, 0] = 0xFFFFFFFF
    elif what == "geom_range":
        sc.tri_geom[-1] = len(sc.geom_material)
    elif what == "geom_order":
        sc.tri_geom[len(sc.tri_geom) // 2 - 1] = 1
        sc.tri_geom[len(sc.tri_geom) // 2] = 0
    elif what == "camera_and_nan":
        sc.camera = sc.camera.copy()
        sc.camera["fovy_deg"] = 200.0
        sc.verts[5, 1] = np.nan
    return sc


@pytest.mark.parametrize("what", ["nan_first", "inf_last", "index_last", "index_max", "geom_range", "geom_order",
                                  "camera_and_nan"])
def test_faulty_meshes_are_refused_as_the_host_check_refuses_them(gpu_device, what):
    good = _soup(3001)
    bad = _bad(good, what)
    print(f"faulty mesh: {what}", flush=True)
    with pytest.raises(wr.WrError) as host:
        wr.validate(bad)
    with pytest.raises(wr.WrError) as gpu:
        wr.GpuScene(gpu_device, bad)
    assert gpu.value.code == host.value.code and str(gpu.value) == str(host.value)
    wr.GpuScene(gpu_device, good).bvh_check(good)


def test_builds_from_several_threads_share_the_handle(gpu_device):
    scs = [_soup(n) for n in (500, 3000, 20_000, 60_000)]
    serial = [wr.GpuScene(gpu_device, sc).bvh_check(sc)["hash"] for sc in scs]
    got = [[] for _ in scs]

    def work(k):
        for _ in range(4):
            gs = wr.GpuScene(gpu_device, scs[k])
            got[k].append(gs.bvh_check(scs[k])["hash"])
            gs.close()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(scs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert got == [[h] * 4 for h in serial]
